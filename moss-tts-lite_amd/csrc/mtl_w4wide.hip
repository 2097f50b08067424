// int4 GEMM at prompt length on the reference's records for gfx950: y[M, N] = x[M, K] @ W,
// W = (q - 8) * scale + zero, for prompts of many rows (the quantized prefill,
// moss_tts_lite/fast.py:218-270).
//
// Why a second GEMM beside mtl_w4prefill.hip.  That kernel multiplies the codes as bf16
// 128 + q and applies scale and zero to each group's sum: two FMAs per output and group, so
// at g = 32 every 16x16x32 MFMA (16 cycles) is followed by 8 VALU instructions (32 cycles),
// and each of its workgroups converts x again.  Here the weights enter the MFMA dequantised
// but for the zero: s * (q - 8) has at most 8 + 3 significant bits and an f16 holds 11, so the
// f16 operand is exact, the accumulators run over all of K with no work per group, and the
// group size matters little.  The zeros add the product of the groups' zeros and x sums, an
// MFMA contraction over 3 K / g (9 % of the main one at g = 32, 2 % at 128).
//
// Measured, both launches, against mtl_w4prefill.hip on one chip: 389 x 4096 x 24576 at g = 32
// 173 -> 98 us (800 TFLOP/s), 1100 x 4096 x 24576 at g = 32 404 -> 253 us, 1536 x 12288 x 4096
// at g = 128 195 -> 157 us (985 TFLOP/s; a large bf16 matrix product of the library reaches
// 1450 here).
//
// Range.  A launch before the GEMM (wide_stage_kernel) finds a power of two per row of x and
// per column of W that puts the largest magnitude of x at 2^6 .. 2^7 and of 8 s and z at
// 2^13 .. 2^14; the result is scaled back exactly.  A bf16 x within 2^23 of its row's maximum
// and a scale or zero within 2^23 of its column's are then exact in f16; smaller ones are cut
// (towards zero) with an absolute error below 2^-24 (x: 2^-30 of the row's maximum, s and z:
// 2^-37 of the column's), under the rounding of the fp32 sums.  X, the fp32 sum of a group's x,
// enters as three f16 parts.  fp32 output against float64, this GEMM and mtl_w4prefill.hip:
// 2.6e-7 and 8.7e-7 at 389 x 4096 x 4096, g = 32, and with one channel in 256 at 2^10 to 2^26
// times the others 3.3e-7 at most and 1.6e-6 to 3e-6.
#include "mtl_w4core.h"
#include "mtl_w4wide_reads.h"

namespace mtl {

typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

constexpr int kWdStrips = 4;                     // 16-column strips per wave
constexpr int kWdCols = 4 * kWdStrips * 16;      // 256 columns per workgroup
constexpr int kWdMaxRT = 6;                      // 16-row tiles per workgroup: 144 KB of LDS
constexpr int kXTop = 6, kWTop = 13;             // binades of the row and column maxima

struct WideArgs {
  const u32x4* xs;            // staged x: [row tile][chunk][lane] (wide_stage_kernel)
  const int32_t* rexp;        // power of two of each row, [16 * row tiles]
  const int32_t* cexp;        // power of two of each column, [N]
  const u32x4* w;             // strip layout
  const uint16_t* sf;         // staged scales f16 [strip][block][column][MB]
  const u32x4* zf;            // staged zeros f16 [strip][32 groups][lane]
  void* y;
  int64_t ldy;
  int M, K, N, kblocks, krec, zchunks, chunks;              // chunks: K/32 + 3 zchunks
  int epilogue, out_f32, rtiles, nb;                        // row tiles, row blocks
  int pack;                   // y and its rows aligned for four results per store
};

struct StageArgs {
  const uint16_t* x;          // bf16 [M, K], rows ldx apart
  u32x4* xs;
  int32_t* rexp;
  int32_t* cexp;
  uint16_t* sf;
  u32x4* zf;
  const uint32_t* qsz;        // (scale, zero) pairs [K/g][N]
  int64_t ldx;
  int M, K, N, group, ngroups, mb, krec, zchunks, chunks, rowblocks;
};

// The exponent that takes a magnitude with bf16 bits b (sign cleared) to binade `top`; 0 for
// zero.  bf16 subnormals count as the smallest normal binade.
__device__ __forceinline__ int top_exp(uint32_t b, int top) {
  const int e = (int)(b >> 7);
  return b == 0 ? 0 : top + 127 - (e > 0 ? e : 1);
}

__device__ __forceinline__ uint32_t pk_f16(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a, b));
}

// One launch per GEMM: the first rowblocks workgroups stage x, 256 threads per row; the others
// reduce and stage the columns' metadata, 64 columns each.  Bound by memory latency: 8.6 us at
// 389 x 4096 and 24576 columns at g = 32 (6.4 MB of x, 25 MB of metadata), 24 us at
// 1536 x 12288 (75 MB); with the row read again for its second use 9.5 and 28, and with a wave
// per row and 2-byte metadata stores the first took 16.8.
//
// A row is used twice: for its largest magnitude, then for its f16 values
// in the order of the MFMA operand: chunk c of 32 channels of row tile t is 1 KB, lane l
// holding row l % 16, channels 32 c + 8 (l / 16) .. + 7 in the pair order of the codes.  The
// four rows of a workgroup are neighbours, so their 16-byte pieces fill 64-byte segments.
// Chunk K/32 + 3 c + p holds part p of the sums of groups 32 c .. 32 c + 31.
__global__ void __launch_bounds__(1024) wide_stage_kernel(StageArgs a) {
  __shared__ uint32_t red[16][64];
  const int t = threadIdx.x, lane = t & 63, wave = wave_id();
  if ((int)blockIdx.x >= a.rowblocks) {
    // 64 columns, 8 groups per wave and turn
    const int col = ((int)blockIdx.x - a.rowblocks) * 64 + lane;
    const int cl = col < a.N ? col : a.N - 1;
    uint32_t mx = 0;
    for (int g0 = 8 * wave; g0 < a.ngroups; g0 += 128) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int g = g0 + i < a.ngroups ? g0 + i : a.ngroups - 1;
        const uint32_t v = a.qsz[(size_t)g * a.N + cl];
        // 8 |s| as bf16 bits (3 binades up), |z|
        const uint32_t s = v & 0x7fffu, z = (v >> 16) & 0x7fffu;
        const uint32_t s8 = s == 0 ? 0u : s + (3u << 7);
        mx = max(mx, max(s8, z));
      }
    }
    red[wave][lane] = mx;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = max(mx, red[i][lane]);
    const int ex = top_exp(mx, kWTop);
    if (col >= a.N) return;
    if (wave == 0) a.cexp[col] = ex;
    const int strip = col >> 4, lj = col & 15;
    u32x4* zs = a.zf + (size_t)strip * a.zchunks * 64 + lj;
    uint16_t* ss = a.sf + ((size_t)strip * a.krec * 16 + lj) * a.mb;
    for (int g0 = 8 * wave; g0 < 32 * a.zchunks; g0 += 128) {
      uint32_t sh[8], zh[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const bool in = g0 + i < a.ngroups;      // zeros pad the last 32 groups
        const uint32_t v = a.qsz[(size_t)(in ? g0 + i : 0) * a.N + col];
        const uint32_t h = pk_f16(ldexpf(__uint_as_float(v << 16), ex),
                                  in ? ldexpf(__uint_as_float(v & 0xffff0000u), ex) : 0.f);
        sh[i] = h & 0xffffu;
        zh[i] = h >> 16;
      }
      zs[(g0 >> 5) * 64 + 16 * ((g0 & 31) >> 3)] =
          u32x4{zh[0] | zh[1] << 16, zh[2] | zh[3] << 16, zh[4] | zh[5] << 16, zh[6] | zh[7] << 16};
      if (a.mb == 4) {                           // ngroups is a multiple of 8
        if (g0 < a.ngroups)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            *reinterpret_cast<u32x2*>(ss + (size_t)(g0 / 4 + h) * 64) =
                u32x2{sh[4 * h] | sh[4 * h + 1] << 16, sh[4 * h + 2] | sh[4 * h + 3] << 16};
      } else if (a.mb == 2) {                    // ngroups is even
#pragma unroll
        for (int h = 0; h < 4; ++h)
          if (g0 + 2 * h < a.ngroups)
            *reinterpret_cast<uint32_t*>(ss + (size_t)(g0 / 2 + h) * 32) = sh[2 * h] | sh[2 * h + 1] << 16;
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (g0 + i < a.ngroups) ss[(size_t)(g0 + i) * 16] = (uint16_t)sh[i];
      }
    }
    return;
  }
  // Four workgroups of 4 rows each fill a row tile's 256-byte segments; they are 8 workgroups
  // apart, so on one XCD, whose L2 joins them.
  const int rw = t >> 8, t4 = t & 255;           // row of the workgroup, thread of its 256
  const int rtile = (blockIdx.x >> 5) * 8 + (blockIdx.x & 7);
  const int row = 16 * rtile + 4 * (((int)blockIdx.x >> 3) & 3) + rw, K = a.K;
  if (rtile >= (a.M + 15) / 16) return;
  const int tile = row >> 4, rl = row & 15;
  u32x4* out = a.xs + (size_t)tile * a.chunks * 64 + rl;
  const int items = K >> 3;                      // 8-channel items; a multiple of 32
  const bool live = row < a.M;                   // rows of the last tile past M stage zeros
  const u32x4* xr = reinterpret_cast<const u32x4*>(a.x + (size_t)(live ? row : a.M - 1) * a.ldx);
  // The row's first 8 x 256 items stay in registers (K <= 16384: all), the rest is read again.
  u32x4 xv[8];
#pragma unroll
  for (int c = 0; c < 8; ++c)
    if (256 * c < items) xv[c] = xr[t4 + 256 * c < items ? t4 + 256 * c : 0];
  uint32_t mx = 0;
  auto take = [&](const u32x4& v) {
    const uint32_t e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) mx = max(mx, max(e[j] & 0x7fffu, (e[j] >> 16) & 0x7fffu));
  };
#pragma unroll
  for (int c = 0; c < 8; ++c)
    if (256 * c < items) take(xv[c]);            // item 0 again where there is none
  for (int i = 2048 + t4; i < items; i += 256) take(xr[i]);
  red[wave][lane] = mx;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) mx = max(mx, red[4 * rw + i][lane]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = max(mx, (uint32_t)__shfl_xor((int)mx, o));
  const int ex = live ? top_exp(mx, kXTop) : 0;
  if (t4 == 0) a.rexp[row] = ex;
  uint16_t* zout = reinterpret_cast<uint16_t*>(out);
  const int per = a.group >> 3;                  // items per group: 4, 8, 16 or 32
  // part p of group g: chunk K/32 + 3 (g / 32) + p, lane quarter (g % 32) / 8, element g % 8
  auto zput = [&](int g, float X) {
    const size_t c = (size_t)(K >> 5) + 3 * (g >> 5);
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const uint32_t h = pk_f16(X, 0.f) & 0xffffu;
      zout[((c + p) * 64 + 16 * ((g & 31) >> 3)) * 8 + (g & 7)] = (uint16_t)h;
      X -= f16_to_f32(h);
    }
  };
  auto put = [&](u32x4 v, int i) {
    const bool in = i < items;                   // whole groups are in or out
    if (!live) v = u32x4{0, 0, 0, 0};
    float sum;
    const u32x4 pv = pair_order_dot(v, sum);
    const uint32_t e[4] = {pv.x, pv.y, pv.z, pv.w};
    uint32_t o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      o[j] = pk_f16(ldexpf(__uint_as_float(e[j] << 16), ex),
                    ldexpf(__uint_as_float(e[j] & 0xffff0000u), ex));
    if (in) out[(size_t)(i >> 2) * 64 + 16 * (i & 3)] = u32x4{o[0], o[1], o[2], o[3]};
    sum = group_sum_valu<4>(sum);
    if (per > 4) sum += dpp_f32<kDppHalfMirror>(sum);
    if (per > 8) sum += dpp_f32<kDppMirror>(sum);
    if (per > 16) sum = xor16_add(sum);
    if (in && (i & (per - 1)) == 0) zput(i / per, ldexpf(sum, ex));
  };
#pragma unroll
  for (int c = 0; c < 8; ++c)
    if (256 * c < items) put(xv[c], t4 + 256 * c);
  for (int i0 = 2048; i0 < items; i0 += 256) put(xr[i0 + t4 < items ? i0 + t4 : 0], i0 + t4);
  for (int g = a.ngroups + t4; g < 32 * a.zchunks; g += 256) zput(g, 0.f);
}

// A word of codes becomes the f16 operand s * (q - 8) in three steps of four independent
// instructions: shifts bring each nibble to mantissa bits 6..9, under the exponent of 16 that is
// 16 + q, and (16 + q) * s - 24 * s rounds once, to a value f16 holds (24 s: 2 + 8 bits).
template <int STEP>
__device__ __forceinline__ void dequant_step(uint32_t w, u32x4& t, uint32_t lo, uint32_t magic,
                                             f16x2_t s, f16x2_t n24) {
  if (STEP == 0) {
    t = u32x4{w << 6, w << 2, w >> 2, w >> 6};
  } else if (STEP == 1) {
    t = u32x4{(t.x & lo) | magic, (t.y & lo) | magic, (t.z & lo) | magic, (t.w & lo) | magic};
  } else {
    uint32_t p[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
    for (int i = 0; i < 4; ++i)
      p[i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(
                                              __builtin_bit_cast(f16x2_t, p[i]), s, n24));
    t = u32x4{p[0], p[1], p[2], p[3]};
  }
  asm volatile("" : "+v"(t.x), "+v"(t.y), "+v"(t.z), "+v"(t.w));   // keeps the step here
}

// Four bf16 results of one row, as one store where rows and base allow it.
__device__ __forceinline__ void put4(uint16_t* p, const uint32_t (&o)[4], int pack) {
  if (pack) {
    *reinterpret_cast<u32x2*>(p) = u32x2{o[0] | o[1] << 16, o[2] | o[3] << 16};
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = (uint16_t)o[i];
  }
}

// 1 KB from a buffer (64 lanes x 16 bytes at voff + soff) straight to LDS at `at` + 16 lane.  In
// asm so that the compiler neither waits for it at the next LDS read nor at a barrier: the
// kernel counts these loads itself (wait_and_barrier).
__device__ __forceinline__ void lds_load16(u32x4 rsrc, uint32_t at, int voff, int soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               ::"s"(at), "v"(voff), "s"(rsrc), "s"(soff) : "memory", "m0");
}

// Waits until at most N of the wave's vector loads are outstanding, then for the workgroup.
template <int N>
__device__ __forceinline__ void wait_and_barrier() {
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
}

// A workgroup owns RT row tiles x 256 columns; wave (kg, wn) multiplies all RT tiles by 64
// columns (4 strips) over part kg of the K blocks.  Either way two waves share a SIMD: KW = 2 is
// a workgroup of 8 waves per CU whose two halves of K meet in LDS at the end, for grids that
// would not give most CUs two workgroups; KW = 1 two independent workgroups of 4 waves, whose
// barriers do not hold each other up.  Halves against whole K, both launches: 1100 x 4096 x 24576
// 282 / 254 us at g = 32 and 251 / 226 at g = 128, 389 rows at g = 32 108 / 101; but
// 1100 x 12288 x 4096 at g = 32, 224 workgroups, 143 / 175.  RT = 6 is what three x buffers leave
// of the LDS: a dequantised operand (12 VALU instructions per 8 codes) feeds 6 MFMAs and an x
// operand 4.  The x tiles come by direct loads into LDS two turns ahead (the staged order is the
// operand order, so there is no conversion and no bank conflict), weights and scales into
// registers three turns ahead.
//
// What bounds it at 1536 x 12288 x 4096, g = 128 (counters of an earlier build of this tile,
// 143 us: 1.97 GHz, MFMA busy 53 % of the cycles, LDS 13 %): the instructions a wave issues.  A
// turn (128 channels per wave) took 2.0 us at RT = 4; 1.2 with the dequantisation left out, 1.2
// with the MFMAs left out, and 1.9 without the x loads.  Two buffers instead of three and weights
// one turn ahead cost 5 %.
template <int RT, int MB, int KW>
__global__ void __launch_bounds__(256 * KW) __attribute__((amdgpu_waves_per_eu(2, 2)))
w4_wide_kernel(WideArgs a) {
  // x tiles of three turns, [tile][chunk of the block][lane] (one tile more at an odd RT, for
  // the halves' exchange at the end)
  constexpr int kBuf = (RT + 1) / 2 * 512;
  __shared__ u32x4 xa[3][KW][kBuf];
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int kg = wave >> 2, wn = wave & 3;
  const int lg = lane >> 4, lj = lane & 15;
  const int N = a.N, kb = a.kblocks;

  // XCD-contiguous tiles, the row blocks of one column tile first: they share its weights
  const int total = (int)gridDim.x, xcd = blockIdx.x & 7, q = total >> 3, rem = total & 7;
  const int id = xcd * q + (xcd < rem ? xcd : rem) + (int)(blockIdx.x >> 3);
  const int ctile = id / a.nb, rb = id - ctile * a.nb;
  const int rbase = a.rtiles / a.nb, rext = a.rtiles - rbase * a.nb;
  const int mt0 = rb * rbase + (rb < rext ? rb : rext);
  const int nrt = rbase + (rb < rext ? 1 : 0);   // <= RT; tiles past it repeat the last one
  const int strip0 = (ctile * 4 + wn) * kWdStrips;

  const uint64_t xbase = reinterpret_cast<uint64_t>(a.xs + (size_t)mt0 * a.chunks * 64);
  const uint32_t xbytes = (uint32_t)(nrt * a.chunks) * 1024u;
  const __amdgpu_buffer_rsrc_t xrsrc = __builtin_amdgcn_make_buffer_rsrc(
      reinterpret_cast<void*>(xbase), (short)0, (int)xbytes, 0x00020000);
  const u32x4 xres{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)xbase),
                   (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(xbase >> 32) & 0xffffu)),
                   (uint32_t)__builtin_amdgcn_readfirstlane((int)xbytes), 0x00020000u};
  const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<u32x4*>(a.w), (short)0, (int)((int64_t)(N / 16) * kb * 1024), 0x00020000);
  const __amdgpu_buffer_rsrc_t srsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(a.sf), (short)0, (int)((int64_t)N * a.krec * MB * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t zrsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<u32x4*>(a.zf), (short)0, (int)((int64_t)(N / 16) * a.zchunks * 1024), 0x00020000);

  // strips past N repeat the last one and are not stored
  int strip[kWdStrips];
#pragma unroll
  for (int s = 0; s < kWdStrips; ++s) strip[s] = wide_strip(strip0 + s, N / 16);
  const int nblk = kb / KW, b0 = kg * nblk;      // this wave group's blocks (kb is even)
  u32x4 wq[3][kWdStrips];
  u32x2 mq[3][kWdStrips];                        // its scales, packed f16 (MB = 4: both words)
  auto issue_w = [&](int r, int i) {             // block i of the group's (clamped)
    const int b = b0 + (i < nblk ? i : nblk - 1);
#pragma unroll
    for (int s = 0; s < kWdStrips; ++s) {
      const int at = wide_scale_at(strip[s], a.krec, kb, b, MB);
      if (MB == 4) {
        mq[r][s] = __builtin_bit_cast(
            u32x2, __builtin_amdgcn_raw_buffer_load_b64(srsrc, lj * 8, at, 0));
      } else if (MB == 2) {
        mq[r][s].x = __builtin_amdgcn_raw_buffer_load_b32(srsrc, lj * 4, at, 0);
      } else {
        mq[r][s].x = __builtin_amdgcn_raw_buffer_load_b16(srsrc, lj * 2, at, 0);
      }
      wq[r][s] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                               wrsrc, lane * 16, wide_weight_at(strip[s], kb, b), 0));
    }
  };
  constexpr int kLoadsW = 2 * kWdStrips;         // loads of one issue_w (in order, as issued)
  // wave wn brings chunk wn of every tile of the block into buffer r
  const uint32_t lds0 = (uint32_t)__builtin_amdgcn_readfirstlane(
      (int)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)&xa[0][kg][64 * wn]);
  const int tstep = a.chunks * 1024;
  auto issue_x = [&](int r, int i) {
    const int b = b0 + (i < nblk ? i : nblk - 1);
    int off = (4 * b + wn) * 1024;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      lds_load16(xres, lds0 + (uint32_t)((r * KW * kBuf + 256 * t) * 16), lane * 16, off);
      if (t + 1 < nrt) off += tstep;
    }
  };
  issue_w(0, 0);
  issue_x(0, 0);
  issue_w(1, 1);
  issue_x(1, 1);
  issue_w(2, 2);

  floatx4 acc[RT][kWdStrips];
  const floatx4 zero4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int tt = 0; tt < RT; ++tt)
#pragma unroll
    for (int s = 0; s < kWdStrips; ++s) acc[tt][s] = zero4;

  // zeros: sum over the groups of z * X, 32 groups per MFMA, X in three parts
  for (int c = kg; c < a.zchunks; c += KW) {
    f16x8_t Z[kWdStrips];
#pragma unroll
    for (int s = 0; s < kWdStrips; ++s)
      Z[s] = __builtin_bit_cast(f16x8_t, __builtin_amdgcn_raw_buffer_load_b128(
          zrsrc, lane * 16, wide_zero_at(strip[s], a.zchunks, c), 0));
    const int k0 = (a.K >> 5) + 3 * c;
#pragma unroll
    for (int tt = 0; tt < RT; ++tt) {
      const int tile = tt < nrt ? tt : nrt - 1;
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        const f16x8_t X = __builtin_bit_cast(f16x8_t, __builtin_amdgcn_raw_buffer_load_b128(
            xrsrc, lane * 16, (tile * a.chunks + k0 + p) * 1024, 0));
#pragma unroll
        for (int s = 0; s < kWdStrips; ++s)
          acc[tt][s] = __builtin_amdgcn_mfma_f32_16x16x32_f16(Z[s], X, acc[tt][s], 0, 0, 0);
      }
    }
  }

  const uint32_t kMagic = vgpr_const(0x4C004C00u);   // f16 (16, 16)
  const uint32_t kLo = vgpr_const(0x03C003C0u);
  u32x4 B[2][kWdStrips];
  // Step g of the 12 that form the operands of chunk j from ring slot r: the strips go two by
  // two through the three steps, so that no instruction waits for the one before it.
  auto piece = [&](int r, int j, int g) {
    const int s = 2 * (g / 6) + (g & 1), step = g % 6 / 2;
    const u32x4 w = wq[r][s];
    const uint32_t word = j == 0 ? w.x : j == 1 ? w.y : j == 2 ? w.z : w.w;
    const int m = MB == 4 ? j : MB == 2 ? j >> 1 : 0;
    const f16x2_t sp = __builtin_bit_cast(f16x2_t, m >> 1 ? mq[r][s].y : mq[r][s].x);
    const _Float16 sc = m & 1 ? sp.y : sp.x;
    const f16x2_t s2{sc, sc};
    const f16x2_t n24 = s2 * f16x2_t{(_Float16)-24.f, (_Float16)-24.f};
    u32x4& t = B[j & 1][s];
    if (step == 0) dequant_step<0>(word, t, kLo, kMagic, s2, n24);
    else if (step == 1) dequant_step<1>(word, t, kLo, kMagic, s2, n24);
    else dequant_step<2>(word, t, kLo, kMagic, s2, n24);
  };
  f16x8_t X[4];
  auto x_frag = [&](int r, int n) {
    return __builtin_bit_cast(f16x8_t, xa[r][kg][(4 * (n % RT) + n / RT) * 64 + lane]);
  };
  // Block i in slot r.  Its first operands are ready; under the MFMAs of chunk j the operands
  // of chunk j + 1 are formed, under chunk 3's those of the next block (slot r1), whose x the
  // last barrier has already covered.
  auto block = [&](int r, int r1, int i) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int tt = 0; tt < RT; ++tt) {
        const int n = j * RT + tt;
        X[(n + 3) & 3] = n + 3 < 4 * RT ? x_frag(r, n + 3) : x_frag(r1, n + 3 - 4 * RT);
#pragma unroll
        for (int s = 0; s < kWdStrips; ++s) {
          acc[tt][s] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
              __builtin_bit_cast(f16x8_t, B[j & 1][s]), X[n & 3], acc[tt][s], 0, 0, 0);
          const int m = 4 * tt + s;              // MFMA of the chunk: steps spread over all
#pragma unroll
          for (int g = 0; g < 12; ++g)
            if (g * 4 * RT / 12 == m) {
              if (j < 3) piece(r, j + 1, g);
              else piece(r1, 0, g);
            }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  };
  // Ends a turn: the block three on is on its way to the registers this turn has read, and the
  // x of the next block but one is in LDS for every wave (only those weights are younger).
  auto turn = [&](int r, int i) {
    asm volatile("" ::: "memory");
    issue_w(r, i + 3);
    __builtin_amdgcn_sched_barrier(0);
    wait_and_barrier<kLoadsW>();
  };
  __builtin_amdgcn_s_waitcnt(0x0F70);            // vmcnt(0), in a form the compiler counts too
  wait_and_barrier<0>();
#pragma unroll
  for (int n = 0; n < 3; ++n) X[n] = x_frag(0, n);
#pragma unroll
  for (int g = 0; g < 12; ++g) piece(0, 0, g);
  // Three turns at a time; past the last block a turn only brings in (clamped) blocks, so the
  // loads in flight at every point are the same on every path and no wait is longer than it
  // has to be.
  for (int i = 0; i < nblk; i += 3) {
    issue_x(2, i + 2);
    block(0, 1, i);
    turn(0, i);
    issue_x(0, i + 3);
    if (i + 1 < nblk) block(1, 2, i + 1);
    turn(1, i + 1);
    issue_x(1, i + 4);
    if (i + 2 < nblk) block(2, 0, i + 2);
    turn(2, i + 2);
  }
  wait_and_barrier<0>();                         // no load into LDS is left

  // KW = 2: the halves meet, wave group kg keeping tiles of its half and handing over the others.
  // acc[tt][s][i] is column 16 (strip0 + s) + 4 lg + i of row 16 (mt0 + tt) + lj.
  constexpr int H0 = (RT + 1) / 2;               // group 0 keeps tiles 0 .. H0 - 1
  const floatx4* theirs = reinterpret_cast<const floatx4*>(&xa[KW == 2 ? 1 - kg : 0][0][0]);
  if constexpr (KW == 2) {
    floatx4* mine = reinterpret_cast<floatx4*>(&xa[kg][0][0]);
#pragma unroll
    for (int tt = 0; tt < RT; ++tt)
      if ((tt >= H0) == (kg == 0)) {
        const int slot = tt >= H0 ? tt - H0 : tt;
#pragma unroll
        for (int s = 0; s < kWdStrips; ++s)
          mine[((wn * H0 + slot) * kWdStrips + s) * 64 + lane] = acc[tt][s];
      }
    __syncthreads();
  }
#pragma unroll
  for (int tt = 0; tt < RT; ++tt) {
    if (KW == 2 && (tt >= H0) != (kg == 1)) continue;
    if (tt >= nrt) continue;
    const int slot = tt >= H0 ? tt - H0 : tt;
    const int row = 16 * (mt0 + tt) + lj;
    const int re = a.rexp[row];
    float v[kWdStrips][4];
#pragma unroll
    for (int s = 0; s < kWdStrips; ++s) {
      const floatx4 o =
          KW == 2 ? theirs[((wn * H0 + slot) * kWdStrips + s) * 64 + lane] : zero4;
      const int col = 16 * (strip0 + s) + 4 * lg;
      const int4 ce = *reinterpret_cast<const int4*>(a.cexp + (col < N ? col : 0));
      const int c4[4] = {ce.x, ce.y, ce.z, ce.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) v[s][i] = ldexpf(acc[tt][s][i] + o[i], -(re + c4[i]));
    }
    if (row >= a.M) continue;
    if (a.epilogue == MTL_EPI_SILU_MUL) {        // strips 0, 1 gate and 2, 3 up of one block
      uint16_t* act = static_cast<uint16_t*>(a.y) + (size_t)row * a.ldy + 8 * strip0 + 4 * lg;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        if (strip0 >= N / 16) continue;
        uint32_t o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = silu_mul_bf16(v[s][i], v[s + 2][i]);
        put4(act + 16 * s, o, a.pack);
      }
      continue;
    }
#pragma unroll
    for (int s = 0; s < kWdStrips; ++s) {
      if (strip0 + s >= N / 16) continue;
      const size_t off = (size_t)row * a.ldy + 16 * (strip0 + s) + 4 * lg;
      if (a.out_f32) {
        float* yf = static_cast<float*>(a.y) + off;
        if (a.pack) {
          *reinterpret_cast<float4*>(yf) = float4{v[s][0], v[s][1], v[s][2], v[s][3]};
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) yf[i] = v[s][i];
        }
        continue;
      }
      uint16_t* yb = static_cast<uint16_t*>(a.y) + off;
      uint32_t o[4];
      if (a.epilogue == MTL_EPI_RESIDUAL) {      // h = bf16(bf16(acc) + h)
        uint32_t h[4];
        if (a.pack) {
          const u32x2 q = *reinterpret_cast<const u32x2*>(yb);
          h[0] = q.x & 0xffffu; h[1] = q.x >> 16; h[2] = q.y & 0xffffu; h[3] = q.y >> 16;
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) h[i] = yb[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = f32_to_bf16(round_bf16(v[s][i]) + bf16_to_f32(h[i]));
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = f32_to_bf16(v[s][i]);
      }
      put4(yb, o, a.pack);
    }
  }
}

static int64_t wide_zchunks(int64_t K, int64_t group) { return (K / group + 31) / 32; }

// The workspace: x fragments, zero fragments, scales, row and column exponents.
struct WideLayout {
  int64_t xs, zf, sf, rexp, cexp, end;
  WideLayout(int64_t M, int64_t K, int64_t N, int64_t group) {
    const int64_t rt = (M + 15) / 16, zc = wide_zchunks(K, group);
    xs = 0;
    zf = rt * (K / 32 + 3 * zc) * 1024;
    sf = zf + N / 16 * zc * 1024;
    rexp = sf + (K / group * N * 2 + 15) / 16 * 16;
    cexp = rexp + rt * 64;
    end = cexp + N * 4;
  }
};

int64_t wide_workspace_bytes(int64_t M, int64_t K, int64_t N, int32_t group) {
  return WideLayout(M, K, N, group).end;
}

// Row blocks: the count that minimises the rounds of workgroups over the CUs times the time of
// a turn at its row tiles (the figures of wide_us).
static double turn_us(int64_t rt) { return rt <= 4 ? 2.3 : rt == 5 ? 2.7 : 3.1; }

static int wide_row_blocks(int64_t rtiles, int64_t ctiles, int cus) {
  int best = 0;
  double cost = 0;
  for (int64_t nb = (rtiles + kWdMaxRT - 1) / kWdMaxRT; nb <= rtiles; ++nb) {
    const int64_t rt = (rtiles + nb - 1) / nb;
    const double c = (double)((nb * ctiles + cus - 1) / cus) * turn_us(rt);
    if (!best || c < cost) { best = (int)nb; cost = c; }
    if (rt <= 4) break;                          // smaller blocks take no less time
  }
  return best;
}

// Estimated time of this GEMM: a turn of 256 channels by its row tiles (0.82 of it at g >= 128,
// with fewer scales), the rounds of workgroups, 14 us for both launches' ends, and the staged
// bytes at about 3 TB/s.
static double wide_us(int64_t M, int64_t K, int64_t N, int32_t group, int cus) {
  const int64_t rtiles = (M + 15) / 16, ctiles = (N + kWdCols - 1) / kWdCols;
  const int64_t nb = wide_row_blocks(rtiles, ctiles, cus);
  return 14.0 + (M * K * 4.0 + K / group * N * 8.0) / 3e6 +
         (double)((nb * ctiles + cus - 1) / cus) * (K / 256) * turn_us((rtiles + nb - 1) / nb) *
             (group >= 128 ? 0.82 : 1.0);
}

// Estimated time of what takes the rows otherwise: the prompt-length GEMM's 64 x 128 tiles (us
// per 4096 channels with the chip full) and its split sums, or, where N is no multiple of
// 128, the skinny GEMM on 16 rows at a time.
static double other_us(int64_t M, int64_t K, int64_t N, int32_t group, int cus) {
  if (N % 128 != 0) return (double)((M + 15) / 16) * (4.0 + K / 4096.0 + K * (double)N / 2.2e7);
  const int64_t tiles = (M + 63) / 64 * (N / 128);
  const double split = (double)(mtl_w4_gemm_prefill_workspace_bytes(M, K, N)) / 2.2e6;
  return 2.0 + tiles * (K / 4096.0) * (group >= 128 ? 0.091 : group == 64 ? 0.105 : 0.1276) +
         (split > 0 ? 4.0 + split : 0.0);
}

// Measured (us, this GEMM / the other, both launches of each, 256 CUs; * where the rule takes it):
//   K x N, g          M = 96     128      192      256      389       600       1100
//   4096 x 24576, 32  48 / 55    48/58*   59/87*   81/96    98/173*   145/234*  253/404*
//   4096 x 24576, 128 40 / 41    41/45*   52/67*   70/69    87/123*   129/167*  226/290*
//   12288 x 4096, 32  106 / 35   107/37   109/47   110/58   110/99    113/131   142/227*
//   12288 x 4096, 128 90 / 28    92/29    93/36    94/43    94/74     96/97     128/163*
//   4096 x 4096, 128  37 / 19    38/21    39/23    40/24    41/34     43/40     53/65*
//   4096 x 5120, 32   43 / 25    45/27    46/29    47/35    47/51     48/71*    66/102*
//   1024 x 2000, 32   19 / 29*   20/39*   20/59*   21/78*   21/121*   22/185*   25/337*
// The line lies where the estimates cross, with a tenth in hand, from 64 rows on.  wide_us counts
// one workgroup per CU in a round, also for the grids that run two (KW = 1), so it errs towards
// the other GEMM: 96 and 256 rows of 4096 x 24576 at g = 32 and 600 of 12288 x 4096 stay there,
// 7 to 18 us slower than here.  No shape of a sweep over 64 to 1536 rows was found slower here.
bool wide_pays(int64_t M, int64_t K, int64_t N, int32_t group) {
  if (M < 64 || M > (1 << 20) || K < 256 || K % 256 != 0 || K > 65536 || N < 16 || N % 16 != 0)
    return false;
  const int64_t cols = (N + kWdCols - 1) / kWdCols * kWdCols;   // offsets stay in 31 bits
  if (cols / 16 * (K / 128) * 1024 >= ((int64_t)1 << 31) || cols * (K / 32) * 4 >= ((int64_t)1 << 31))
    return false;
  const int cus = pf_device_cus();
  return 1.1 * wide_us(M, K, N, group, cus) < other_us(M, K, N, group, cus);
}

template <int MB, int KW>
static void wide_launch(const WideArgs& a, dim3 grid, int rt, hipStream_t st) {
  const dim3 block(256 * KW);
  switch (rt) {
    case 6: hipLaunchKernelGGL((w4_wide_kernel<6, MB, KW>), grid, block, 0, st, a); break;
    case 5: hipLaunchKernelGGL((w4_wide_kernel<5, MB, KW>), grid, block, 0, st, a); break;
    default: hipLaunchKernelGGL((w4_wide_kernel<4, MB, KW>), grid, block, 0, st, a); break;
  }
}

int wide_gemm(const void* x, int64_t M, int64_t ldx, int64_t K, const int32_t* strip_weight,
              const void* qsz, int64_t N, int32_t group, int32_t epilogue, bool out_f32, void* y,
              int64_t ldy, void* workspace, hipStream_t st) {
  const int64_t rtiles = (M + 15) / 16;
  StageArgs s;
  s.x = static_cast<const uint16_t*>(x);
  s.qsz = static_cast<const uint32_t*>(qsz);
  s.ldx = ldx;
  s.M = (int)M; s.K = (int)K; s.N = (int)N;
  s.group = group;
  s.ngroups = (int)(K / group);
  s.zchunks = (int)wide_zchunks(K, group);
  s.chunks = (int)(K / 32) + 3 * s.zchunks;
  s.rowblocks = (int)(rtiles + 7) / 8 * 32;
  s.mb = group >= 128 ? 1 : 128 / group;
  s.krec = (int)(K / (group > 128 ? 256 : 128));
  const WideLayout lay(M, K, N, group);
  char* const ws = static_cast<char*>(workspace);
  s.xs = reinterpret_cast<u32x4*>(ws + lay.xs);
  s.zf = reinterpret_cast<u32x4*>(ws + lay.zf);
  s.sf = reinterpret_cast<uint16_t*>(ws + lay.sf);
  s.rexp = reinterpret_cast<int32_t*>(ws + lay.rexp);
  s.cexp = reinterpret_cast<int32_t*>(ws + lay.cexp);
  hipLaunchKernelGGL(wide_stage_kernel, dim3((unsigned)(s.rowblocks + (N + 63) / 64)), dim3(1024), 0,
                     st, s);
  WideArgs a;
  a.xs = s.xs; a.rexp = s.rexp; a.cexp = s.cexp;
  a.w = reinterpret_cast<const u32x4*>(strip_weight);
  a.sf = s.sf;
  a.zf = s.zf;
  a.y = y;
  a.ldy = ldy;
  a.M = s.M; a.K = s.K; a.N = s.N;
  a.kblocks = (int)(K / 128);
  a.krec = s.krec;
  a.zchunks = s.zchunks;
  a.chunks = s.chunks;
  a.epilogue = epilogue;
  a.out_f32 = out_f32;
  a.rtiles = (int)rtiles;
  a.pack = ldy % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & (out_f32 ? 15u : 7u)) == 0;
  const int64_t ctiles = (N + kWdCols - 1) / kWdCols;
  a.nb = wide_row_blocks(rtiles, ctiles, pf_device_cus());
  const int rt = (int)((rtiles + a.nb - 1) / a.nb);
  const dim3 grid((unsigned)(a.nb * ctiles));
  const bool two = 2 * (int64_t)grid.x < 3 * pf_device_cus();   // one workgroup for most CUs
  if (s.mb == 1) two ? wide_launch<1, 2>(a, grid, rt, st) : wide_launch<1, 1>(a, grid, rt, st);
  else if (s.mb == 2) two ? wide_launch<2, 2>(a, grid, rt, st) : wide_launch<2, 1>(a, grid, rt, st);
  else two ? wide_launch<4, 2>(a, grid, rt, st) : wide_launch<4, 1>(a, grid, rt, st);
  return launch_status();
}

}  // namespace mtl

using namespace mtl;

extern "C" {

int64_t mtl_w4_gemm_prompt_qsz_workspace_bytes(int64_t M, int64_t K, int64_t N,
                                               int32_t group_size) {
  if (group_size != 32 && group_size != 64 && group_size != 128 && group_size != 256) return 0;
  return wide_pays(M, K, N, group_size) ? wide_workspace_bytes(M, K, N, group_size) : 0;
}

int mtl_w4_gemm_prompt_qsz(const void* x, int64_t M, int64_t ldx, int64_t K,
                           const int32_t* strip_weight, const void* qsz, int64_t N,
                           int32_t group_size, int32_t epilogue, int32_t out_dtype, void* y,
                           int64_t ldy, void* workspace, int64_t ws_bytes, void* stream) {
  if (!x || !strip_weight || !qsz || !y) return MTL_ERR_INVALID_ARG;
  if (epilogue != MTL_EPI_NONE && epilogue != MTL_EPI_RESIDUAL && epilogue != MTL_EPI_SILU_MUL)
    return MTL_ERR_INVALID_ARG;
  if (out_dtype != MTL_OUT_BF16 && out_dtype != MTL_OUT_F32) return MTL_ERR_INVALID_ARG;
  if (epilogue != MTL_EPI_NONE && out_dtype != MTL_OUT_BF16) return MTL_ERR_INVALID_ARG;
  if (group_size != 32 && group_size != 64 && group_size != 128 && group_size != 256)
    return MTL_ERR_GROUP;
  const int64_t ncols = epilogue == MTL_EPI_SILU_MUL ? N / 2 : N;
  const int64_t cols = (N + kWdCols - 1) / kWdCols * kWdCols;
  if (M < 1 || M > (1 << 20) || K <= 0 || K % 256 != 0 || K > 65536 || N <= 0 || N % 16 != 0 ||
      N > ((int64_t)1 << 30) || (epilogue == MTL_EPI_SILU_MUL && N % 64 != 0) ||
      K % group_size != 0 || ldx < K || ldy < ncols ||
      cols / 16 * (K / 128) * 1024 >= ((int64_t)1 << 31) ||
      cols * (K / 32) * 4 >= ((int64_t)1 << 31))
    return MTL_ERR_SHAPE;
  if (!aligned16(x) || ldx % 8 != 0 || !aligned16(strip_weight) ||
      (reinterpret_cast<uintptr_t>(qsz) & 3u) ||
      (reinterpret_cast<uintptr_t>(y) & (out_dtype == MTL_OUT_F32 ? 3u : 1u)))
    return MTL_ERR_ALIGN;
  if (!workspace || ws_bytes < wide_workspace_bytes(M, K, N, group_size)) return MTL_ERR_WORKSPACE;
  if (!aligned16(workspace)) return MTL_ERR_ALIGN;
  return wide_gemm(x, M, ldx, K, strip_weight, qsz, N, group_size, epilogue,
                   out_dtype == MTL_OUT_F32, y, ldy, workspace, (hipStream_t)stream);
}

}  // extern "C"
