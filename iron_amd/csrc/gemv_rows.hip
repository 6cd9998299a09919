// Weight-streaming int8 GEMV for batches up to 15 on the fp64 matrix instructions of gfx950:
//   y[b][m] = EPI( sum_k q[m][k] s[m][k / G] x[b][k] )
//
// Reference: the arithmetic of the batch-1 kernel (gemv.hip): the golden GEMVInt8.reference
// (iron/operators/gemv_int8/op.py:173-178) on the row-block wire of gemv_int8/reference.py:59-80,
// every product exact, accumulated in fp64 and rounded once by the epilogue.
//
// Mapping: v_mfma_f64_4x4x4 multiplies four independent 4x4 blocks: lane l holds A[row l % 4] and
// B[column l % 4] of block (l / 4) % 4 at k (l / 16), and D[row l / 16][column l % 4] of that block
// (layout checked on the device). Rows are weight rows, columns batch rows, and the 16 (block, k)
// positions are 16 slices of a 256-wide K chunk: a lane multiplies 16 consecutive weights of one
// row with the 16 matching x values of one batch row, element j of every lane's slice in step j
// of 16. The blocks' sums add at the end of a row tile. x is spread over the lanes (no lane holds
// another batch row's copy), so a batch of four costs 16 x values per lane where the vector form
// held 64.
//
// Neighbouring lanes belong to different rows, and a load in that order costs a cache access per
// lane (64 clocks; 16 x that pattern made the loads alone 39 us of an LM head). So a load reads 16
// lanes x 16 bytes of one row, and the step passes through LDS: written in load order, read back
// in operand order, 16-byte pieces XOR-swizzled by row so that neither side has bank conflicts
// (wavefront-private, no barrier).
//
// A weight becomes its fp64 value q s in two instructions: v_perm_b32 puts the biased byte
// u = q + 128 into the high word of 4096 + u, and fma(4096 + u, s, -4224 s) = q s exactly (a
// 21-bit product). An infinite scale makes that inf - inf, and its row's outputs NaN: a NaN output is
// set aside and summed again at the end, each 16-weight slice of q x before its scale as in the batch-1
// kernel (a look at the scales in every step cost 2 %, the sum beside the store 1 %).
//
// A workgroup of 8 wavefronts owns a contiguous run of row tiles (4 R rows); its (tile, K chunk)
// steps are cut into 8 contiguous ranges, one per wavefront, so every wavefront has the same work
// to within a step whatever M and K are. A wavefront that covers a whole tile finishes it alone;
// the partial sums of a tile that spans wavefronts meet in LDS and add in wavefront order. Loads
// run a step or two ahead in registers (weights, scales and x of a step together: vector
// loads complete in issue order). 256 workgroups at most: one per CU, each streaming its share (with
// few tiles, one for each column group of a share).
//
// What bounds it: instruction issue, most of it on the fp64 pipe, which the matrix and vector forms
// share. Per 64 weights a v_mfma_f64_4x4x4 takes 16 clocks per four batch rows, the dequantizing fma
// about 5 and the byte permute 4. Measured, us, HBM-cold, before (a vector FMA per weight and batch
// row, one row group per workgroup) and now:
//   4096 x 12288, G = 128, B = 12 / 4         187 / 96          33 / 18         (10 us of HBM reads)
//   1024 x 1024, B = 3 / 5 / 12               3.8 / 5.1 / 7.2   3.8 / 4.3 / 4.7
//   1024 x 512, G = 16, B = 5 / 15            3.8 / 5.2         3.9 / 4.6
//   64 x 16384, B = 5 / 15                    12.0 / 12.1       10.8 / 10.8
//   151936 x 1024 with argmax, G = 32, B = 4  106               50              (33 us)
//   Qwen3-4B at B = 3: QKV 6144 x 2560        24                12
//     Wo 2560 x 4096                          12                8
//     gate/up 2 x 9728 x 2560                 51                22
//     down 2560 x 9728                        37                13
// The same loop without the matrix products (timing only) takes 37 us on the LM head. A wavefront
// raises its priority while it converts (the SIMD's other one then issues its products: 50.8 ->
// 49.2 us on the head).
#include <type_traits>

#include "common.h"
#include "gemv_core.h"
#include "internal.h"

namespace {

using namespace iron::dev;

constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr int kChunk = 256;    // K elements per step: 16 per lane and row
constexpr int kCUs = 256;
// LDS columns of staged x: 64 16-byte units (a chunk) + 4, so the 16 units that 16 lanes read
// (4 columns x 4 slices) fall on distinct banks
constexpr int kColUnits = 68;
constexpr int kMaxLds = 163840 - 1024;
constexpr int kMaxB = 16;

// Where a step's x comes from: bf16 or fp32 rows in memory, or fp32 values staged in LDS (the
// RMSNorm prologues, computed once per workgroup)
enum XSrc : int { X_BF16 = 0, X_F32 = 1, X_LDS = 2 };

// 4 bytes at an even address (two scales)
typedef uint32_t __attribute__((aligned(2))) pair16_t;
// A load at a wave-uniform base plus a 32-bit lane offset.
template <class T>
IRON_DEV T ld_at(const uint8_t* base, uint32_t off) {
  return *(const __attribute__((address_space(1))) T*)(
      (const __attribute__((address_space(1))) uint8_t*)base + off);
}

// A launch's shares, worked out on the host: T row tiles are `tiles` per workgroup and `extra` more
// (0 for fewer workgroups than kCUs), spread evenly: workgroup b's begin at b T / kCUs. scales: a wire
// block's payload bytes (its scale run starts there).
struct Shares {
  int tiles, extra;
  size_t scales;
};

// Batch rows [b0, b0 + n) of a call: operands advanced by b0 rows.
__host__ __device__ inline GemvParams rows_of(const GemvParams& p, int b0, int n) {
  GemvParams q = p;
  q.nb = n;
  if (p.pro == PRO_F32) q.x = (const float*)p.x + (size_t)b0 * p.x_stride;
  else q.x = (const uint16_t*)p.x + (size_t)b0 * p.x_stride;
  if (p.x2) q.x2 = p.x2 + (size_t)b0 * p.x2_stride;
  if (p.epi == EPI_F32 || p.epi == EPI_SWIGLU_F32) q.y = (float*)p.y + (size_t)b0 * p.y_stride;
  else q.y = (uint16_t*)p.y + (size_t)b0 * p.y_stride;
  if (p.r1) q.r1 = p.r1 + (size_t)b0 * p.r_stride;
  if (p.r2) q.r2 = p.r2 + (size_t)b0 * p.r_stride;
  if (p.argmax) q.argmax = p.argmax + b0;
  return q;
}

// G16: quantization groups of 16 (twice the scales per chunk). kDepth: steps in flight. kSplit: a
// workgroup takes one group of four batch rows (blockIdx.y).
template <int NB, int R, bool DUAL, int XS, bool G16, int kDepth, bool kSplit = false>
__global__ __launch_bounds__(kThreads) void gemv_rows_kernel(GemvParams p, Shares share) {
  if constexpr (kSplit) p = rows_of(p, 4 * (int)blockIdx.y, min(p.nb - 4 * (int)blockIdx.y, 4));
  constexpr int NM = DUAL ? 2 : 1;
  constexpr int TR = 4 * R;                                      // rows per tile
  constexpr int NS = G16 ? 2 : 1;                                // scale dwords per lane
  constexpr int XR = XS == X_BF16 ? 2 : (XS == X_F32 ? 4 : 1);   // 16-byte x pieces per column
  extern __shared__ float4 s_x[];                                // X_LDS: [chunk][nb] columns
  // sums of the tiles a wavefront shares: [0] one begun by an earlier wavefront, [1] its own last
  __shared__ double s_part[kWaves][2][NM][NB * 4][TR];
  struct StepLds {
    iron_u32x4 w[NM * R * 64];
    iron_u32x4 x[XS == X_LDS ? 1 : NB * XR * 64];
    uint32_t sc[NM * 64 * NS];
  };
  __shared__ __align__(16) StepLds s_step[kWaves];
  __shared__ unsigned long long s_best[kMaxB];
  __shared__ double s_ss[4][2];

  const int tid = threadIdx.x, lane = tid & 63;
  // Wavefronts go to the four SIMDs in turn. In this order neighbours share one, so that the ranges of
  // a workgroup with fewer steps than wavefronts (every eighth, fourth or second) fall on different
  // SIMDs.
  const int hw = __builtin_amdgcn_readfirstlane(tid >> 6), wave = (hw & 3) * 2 + (hw >> 2);
  const int sub = lane & 3, slot = lane >> 2;  // A row / B column, slice of the chunk
  const int K = p.K, nb = p.nb;
  const int C = (K + kChunk - 1) / kChunk;
  auto first = [&](int b) { return b * share.tiles + b * share.extra / kCUs; };
  const int t0 = first((int)blockIdx.x), nt = first((int)blockIdx.x + 1) - t0;
  const int S = nt * C;
  auto range = [&](int w) { return S * w / kWaves; };  // S < 2^28 (host check)
  const int s0 = range(wave), s1 = range(wave + 1);

  struct Step {
    iron_u32x4 w[NM][R];
    uint32_t sc[NM][NS];
    iron_u32x4 x[NB][XR];
  };
  Step ring[kDepth];
  // Addresses: 32-bit lane offsets from the workgroup's first row, which change with the tile, and
  // scalar bases that advance with the chunk (a load then costs an instruction or two).
  // Load r of the weights: lane l the 16-byte slice l % 16 of row 4 r + l / 16; scales: 4 bytes
  // (two groups) of row l / 4, dword l % 4 (+ 4 for G = 16) of the chunk's scale run. A scale dword
  // may begin a group ahead of its run (below), so its base does, and its offset counts from there.
  const int ng = K >> p.gshift;
  const uint32_t blk0 = fastdiv((uint32_t)(t0 * TR), p.tdiv);
  const uint32_t in0 = (uint32_t)(t0 * TR) - blk0 * (uint32_t)p.tile_m;
  const size_t wbase = wire_row_base(blk0, p.blk_bytes, 0, in0, (uint32_t)K);
  const size_t sbase =
      wire_row_base(blk0, p.blk_bytes, share.scales, in0, 2u * (uint32_t)ng) - 2;
  const uint8_t *wp[NM], *sp[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    wp[m] = (m ? p.w2 : p.w) + wbase;
    sp[m] = (m ? p.w2 : p.w) + sbase;
  }
  uint32_t woff[R], soff;
  auto aim = [&](int tile) __attribute__((always_inline)) {
    auto offset_of = [&](int in_tile, uint32_t row_bytes) {
      const uint32_t row = (uint32_t)min((t0 + tile) * TR + in_tile, p.M - 1);
      const uint32_t blk = fastdiv(row, p.tdiv);
      return wire_row_offset(blk - blk0, p.blk_bytes, row - blk * (uint32_t)p.tile_m, in0,
                             row_bytes);
    };
#pragma unroll
    for (int r = 0; r < R; ++r) woff[r] = offset_of(4 * r + (lane >> 4), (uint32_t)K);
    soff = 2u + offset_of(min(lane >> 2, TR - 1), 2u * (uint32_t)ng);
  };
  constexpr int PC = XS == X_BF16 ? 32 : 64;  // 16-byte x pieces of a column's chunk
  constexpr int PE = kChunk / PC;             // elements per piece
  constexpr int XB = XS == X_BF16 ? 2 : 4;    // bytes per element
  uint32_t xoff[NB * XR];
#pragma unroll
  for (int h = 0; h < NB * XR; ++h)
    xoff[h] = (uint32_t)min((h * 64 + lane) / PC, nb - 1) * (uint32_t)p.x_stride * XB;
  // The loads of a chunk of the tile aimed at. Nothing is conditional (slices past K take an
  // earlier one, rows past M the last row), so that the wait counts stay exact; x past K is zeroed
  // where it is used, rows past M are never stored.
  auto load = [&](Step& g, int chunk) __attribute__((always_inline)) {
    const int k0 = chunk * kChunk, left = K - k0;  // left >= 16
    const uint32_t ks = (uint32_t)min((lane & 15) * 16, left - 16);
    const int g0 = k0 >> p.gshift;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int m = 0; m < NM; ++m)
        g.w[m][r] = ld_at<iron_u32x4>(wp[m] + k0, woff[r] + ks);
#pragma unroll
    for (int q = 0; q < NS; ++q) {
      const int so = min(4 * ((lane & 3) + 4 * q), 2 * (ng - g0) - 4);  // -2 with one group left
#pragma unroll
      for (int m = 0; m < NM; ++m)
        g.sc[m][q] = ld_at<pair16_t>(sp[m] + 2 * g0, soff + (uint32_t)so);
    }
    if constexpr (XS != X_LDS) {
#pragma unroll
      for (int h = 0; h < NB * XR; ++h) {
        const uint32_t kx = (uint32_t)min((h * 64 + lane) % PC * PE, left - PE) * XB;
        g.x[h / XR][h % XR] =
            ld_at<iron_u32x4>((const uint8_t*)p.x + (size_t)k0 * XB, xoff[h] + kx);
      }
    }
  };
  // the next step to load; past the range the last one again
  int ls = s0, lt = s0 / C, lc = s0 - lt * C;
  auto advance = [&]() __attribute__((always_inline)) {
    if (ls + 1 < s1) {
      ++ls;
      if (++lc == C) {
        lc = 0;
        aim(++lt);
      }
    }
  };

  // ---- RMSNorm prologues: hf (fp32) or hn (bf16) of every batch row into LDS. Wavefront w owns
  // row w (two wavefronts per row up to four rows); its inputs are loaded ahead of the first
  // weights, so that their wait does not include the weights'.
  constexpr int U = 64 / kWaves;
  const int wpr = nb <= 4 ? 2 : 1;
  const int part = wpr == 2 ? (hw & 1) : 0;
  const int n8 = K >> 3;
  uint4 xa[XS == X_LDS ? U : 1], xb[XS == X_LDS ? U : 1], xw[XS == X_LDS ? U : 1];
  auto piece = [&](int u) { return part * 64 + lane + 64 * wpr * u; };
  const bool has_x2 = p.x2 != nullptr;
  auto load_row = [&](int b) {
    const uint4* src = (const uint4*)((const uint16_t*)p.x + (size_t)b * p.x_stride);
    const uint4* src2 = has_x2 ? (const uint4*)(p.x2 + (size_t)b * p.x2_stride) : src;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = piece(u) < n8 ? piece(u) : 0;
      if (64 * wpr * u < n8) {  // uniform
        xa[u] = src[i];
        xb[u] = src2[i];
        xw[u] = ((const uint4*)p.nw)[i];
      }
    }
  };
  if constexpr (XS == X_LDS) {
    const int b = wpr == 2 ? hw >> 1 : hw;
    if (b < nb) load_row(b);
  }
  if (s0 < s1) {
    aim(lt);
#pragma unroll
    for (int u = 0; u < kDepth; ++u) {
      load(ring[u], lc);
      __builtin_amdgcn_sched_barrier(0);
      advance();
    }
  }
  if constexpr (XS == X_LDS) {
    const bool to_bf16 = p.pro == PRO_RMS_BF16;
    auto put = [&](int b, int i, double inv, const uint4 a, const uint4 a2, const uint4 w8) {
      float f[8], wf[8];
      slot_values(a, a2, has_x2, f);
      unpack8(w8, wf);
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const double y = ((double)f[j] * inv) * (double)wf[j];
        v[j] = to_bf16 ? round_bf16((float)y) : (float)y;
      }
      const int k = 8 * i, in = k & (kChunk - 1);
      float4* d = s_x + ((size_t)(k / kChunk) * nb + b) * kColUnits + ((in >> 2) & 3) * 16 +
                  (in >> 4);
      d[0] = make_float4(v[0], v[1], v[2], v[3]);
      d[16] = make_float4(v[4], v[5], v[6], v[7]);
    };
    auto square = [&](const uint4 a, const uint4 a2) {
      float f[8];
      slot_values(a, a2, has_x2, f);
      double v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = f[j];
      return sum_sq_tree(v);
    };
    for (int b = wpr == 2 ? hw >> 1 : hw; b < (wpr == 2 ? 4 : nb); b += wpr == 2 ? 4 : kWaves) {
      const bool on = b < nb;  // wave-uniform; with two wavefronts per row all meet at the barrier
      if (on && wpr == 1 && b != hw) load_row(b);
      const uint4* src = (const uint4*)((const uint16_t*)p.x + (size_t)(on ? b : 0) * p.x_stride);
      const uint4* src2 =
          has_x2 ? (const uint4*)(p.x2 + (size_t)(on ? b : 0) * p.x2_stride) : src;
      double ss = 0.0;
      if (on) {
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (piece(u) < n8) ss += square(xa[u], xb[u]);
        for (int i = piece(U); i < n8; i += 64 * wpr) ss += square(src[i], src2[i]);
      }
      ss = wave_sum_d(ss);
      if (wpr == 2) {
        if (lane == 0) s_ss[b][part] = ss;
        __syncthreads();
        ss = s_ss[b][0] + s_ss[b][1];
      }
      if (!on) continue;
      const double inv = inv_rms(ss, K, (double)p.eps);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (piece(u) < n8) put(b, piece(u), inv, xa[u], xb[u], xw[u]);
      for (int i = piece(U); i < n8; i += 64 * wpr)
        put(b, i, inv, src[i], src2[i], ((const uint4*)p.nw)[i]);
    }
    // the last chunk's columns past K
    const int pad0 = (K & (kChunk - 1)) / 16;
    if (pad0) {
      for (int i = tid; i < nb * 64; i += kThreads)
        if ((i & 15) >= pad0)
          s_x[((size_t)(C - 1) * nb + (i >> 6)) * kColUnits + (i & 63)] =
              make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  if (tid < kMaxB) s_best[tid] = 0ull;
  __syncthreads();

  double acc[NM][R][NB];
  auto clear = [&]() {
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int n = 0; n < NB; ++n) acc[m][r][n] = 0.0;
  };
  clear();
  const uint32_t to_u = p.xor_mask ^ 0x80808080u;  // stored bytes -> u = q + 128
  auto compute = [&](Step& g, int chunk) __attribute__((always_inline)) {
    // through LDS from load order to operand order
    iron_u32x4* const lw = s_step[wave].w;
    uint32_t* const ls4 = s_step[wave].sc;
    iron_u32x4* const lx = s_step[wave].x;
    __builtin_amdgcn_wave_barrier();
    {
      const int lr = lane >> 4;
#pragma unroll
      for (int m = 0; m < NM; ++m) {
#pragma unroll
        for (int r = 0; r < R; ++r)
          lw[((m * R + r) * 4 + lr) * 16 + ((lane & 15) ^ (4 * lr))] = g.w[m][r];
#pragma unroll
        for (int q = 0; q < NS; ++q) ls4[((m * 16) + (lane >> 2)) * 4 * NS + 4 * q + (lane & 3)] = g.sc[m][q];
      }
    }
    if constexpr (XS != X_LDS) {
#pragma unroll
      for (int h = 0; h < NB * XR; ++h) {
        const int f = h * 64 + lane, c = f / PC, pc = f % PC;
        const bool in = chunk * kChunk + pc * PE < K;
        lx[c * PC + (pc ^ (XS == X_BF16 ? 4 * (c & 3) : (c & 3)))] =
            in ? g.x[h / XR][h % XR] : iron_u32x4{0u, 0u, 0u, 0u};
      }
    }
    __builtin_amdgcn_wave_barrier();
    iron_u32x4 w[NM][R];
    double sc[NM][R], off[NM][R];
    {
      // this slice's group in the chunk; an odd scale run's last one sits in a high half
      const int gl = (slot * 16) >> p.gshift, e = 2 * ((K >> p.gshift) - ((chunk * kChunk) >> p.gshift));
      const int gb = 2 * min(gl, (e >> 1) - 1) + (((e & 2) && 2 * gl >= e - 2) ? 2 : 0);
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int r = 0; r < R; ++r) {
          w[m][r] = lw[((m * R + r) * 4 + sub) * 16 + (slot ^ (4 * sub))];
          const uint32_t h = ls4[(m * 16 + 4 * r + sub) * 4 * NS + (gb >> 2)];
          sc[m][r] = (double)((gb & 2) ? bf16hi_to_f32(h) : bf16lo_to_f32(h));
          off[m][r] = -4224.0 * sc[m][r];
        }
    }
    const float4* xc[NB];
    if constexpr (XS == X_LDS) {
#pragma unroll
      for (int n = 0; n < NB; ++n)
        xc[n] = s_x + ((size_t)chunk * nb + min(4 * n + sub, nb - 1)) * kColUnits + slot;
    }
    auto xpiece = [&](int n, int pc) {  // 16-byte piece of column 4 n + sub
      return lx[(4 * n + sub) * PC + (pc ^ (XS == X_BF16 ? 4 * sub : sub))];
    };
#pragma unroll
    for (int jq = 0; jq < 4; ++jq) {
      float xf[NB][4];
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        if constexpr (XS == X_BF16) {
          const iron_u32x4 v = xpiece(n, 2 * slot + (jq >> 1));
          const uint32_t a = v[(jq & 1) * 2], c = v[(jq & 1) * 2 + 1];
          xf[n][0] = bf16lo_to_f32(a);
          xf[n][1] = bf16hi_to_f32(a);
          xf[n][2] = bf16lo_to_f32(c);
          xf[n][3] = bf16hi_to_f32(c);
        } else if constexpr (XS == X_F32) {
          const iron_u32x4 v = xpiece(n, 4 * slot + jq);
#pragma unroll
          for (int e = 0; e < 4; ++e) xf[n][e] = __uint_as_float(v[e]);
        } else {
          const float4 v = xc[n][jq * 16];
          xf[n][0] = v.x;
          xf[n][1] = v.y;
          xf[n][2] = v.z;
          xf[n][3] = v.w;
        }
      }
      uint32_t d[NM][R];
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int r = 0; r < R; ++r) d[m][r] = w[m][r][jq] ^ to_u;
      // every conversion of the quad first, then its products: alternating fp64 vector and matrix
      // instructions costs a quarter more (32.5 against 26.2 clocks per 64 weights at one column
      // group, 65 against 58 at three; register-only loop, two wavefronts per SIMD)
      __builtin_amdgcn_s_setprio(1);
      double bx[4][NB], a[4][NM][R];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int n = 0; n < NB; ++n) bx[e][n] = (double)xf[n][e];
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
          for (int r = 0; r < R; ++r) {
            // 4096 + u: u in bits 8..15 of the high word
            const uint32_t hi =
                __builtin_amdgcn_perm(d[m][r], 0x40B00000u, 0x03020000u | ((4u + e) << 8));
            a[e][m][r] = fma(__hiloint2double((int)hi, 0), sc[m][r], off[m][r]);
          }
      }
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(0);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
          for (int r = 0; r < R; ++r)
#pragma unroll
            for (int n = 0; n < NB; ++n)
              acc[m][r][n] =
                  __builtin_amdgcn_mfma_f64_4x4x4f64(a[e][m][r], bx[e][n], acc[m][r][n], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // the epilogue of the call's kind: gate/up (SwiGLU, fp32), down (fp32 x: residual), else bf16,
  // with the argmax key when asked for
  auto store = [&](int row, int col, double v, double v2) __attribute__((always_inline)) {
    const size_t o = (size_t)col * p.y_stride + row;
    if constexpr (DUAL) {
      ((float*)p.y)[o] = (float)silu_mul(v, v2);
    } else if constexpr (XS == X_F32) {
      const size_t ro = (size_t)col * p.r_stride + row;
      float x1 = bf16_to_f32(p.r1[ro]);
      if (p.r2) x1 = x1 + bf16_to_f32(p.r2[ro]);
      ((uint16_t*)p.y)[o] = f64_to_bf16((double)x1 + v);
    } else {
      const uint16_t h = f64_to_bf16(v);
      ((uint16_t*)p.y)[o] = h;
      if (p.epi == EPI_BF16_ARGMAX)
        atomicMax(&s_best[col], ((unsigned long long)bf16_order_key(h) << 32) |
                                    (unsigned long long)(~(uint32_t)row));
    }
  };
  bool aside = false;  // a NaN among this lane's outputs
  auto finish = [&](int row, int col, double v, double v2) __attribute__((always_inline)) {
    if (v == v && v2 == v2) store(row, col, v, v2);
    else aside = true;
  };
  // The outputs of the tile whose sums are at s_part[wave][from], plus the shares of the
  // wavefronts after it whose ranges begin before step `end` (in order).
  auto emit = [&](int tile, int from, int end) __attribute__((always_inline)) {
    for (int o = lane; o < TR * NB * 4; o += 64) {
      const int rt = o % TR, col = o / TR, row = (t0 + tile) * TR + rt;
      double v[NM];
#pragma unroll
      for (int m = 0; m < NM; ++m) v[m] = s_part[wave][from][m][col][rt];
      for (int w = wave + 1; w < kWaves && range(w) < end; ++w) {
        if (range(w) == range(w + 1)) continue;
#pragma unroll
        for (int m = 0; m < NM; ++m) v[m] += s_part[w][0][m][col][rt];
      }
      if (row < p.M && col < nb) finish(row, col, v[0], v[NM - 1]);
    }
  };
  // The end of a tile, or of this wavefront's range: the blocks' sums (lanes l, l ^ 4, l ^ 8 of a
  // 16-lane row) go to LDS; a tile that was wholly this wavefront's own is finished from there (a
  // wavefront's LDS accesses complete in order). Lane (row i = l / 16, column sub) writes the
  // results (r, n) whose index is its block mod 4.
  auto flush = [&](int step, int chunk) __attribute__((always_inline)) {
    const bool begun = step - chunk >= s0;
    const int blk = slot & 3, i = lane >> 4;
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int n = 0; n < NB; ++n) {
          double v = acc[m][r][n];
          v += dpp_d<0x124>(v);  // row_ror:4
          v += dpp_d<0x128>(v);  // row_ror:8
          if (((r * NB + n) & 3) == blk) s_part[wave][begun][m][4 * n + sub][4 * r + i] = v;
        }
    clear();
    if (begun && chunk == C - 1) {
      __builtin_amdgcn_wave_barrier();
      emit((step - chunk) / C, 1, 0);
      __builtin_amdgcn_wave_barrier();
    }
  };

  if (s0 < s1) {
    int cs = s0, cc = s0 % C;
    auto step = [&](Step& g) __attribute__((always_inline)) {
      compute(g, cc);
      if (cc == C - 1 || cs == s1 - 1) flush(cs, cc);
      ++cs;
      if (++cc == C) cc = 0;
      __builtin_amdgcn_sched_barrier(0);
    };
    // whole rounds of the ring, every slot refilled with a step of the range
    for (int it = (s1 - s0) / kDepth - 1; it > 0; --it) {
#pragma unroll
      for (int u = 0; u < kDepth; ++u) {
        step(ring[u]);
        load(ring[u], lc);
        __builtin_amdgcn_sched_barrier(0);
        advance();
      }
    }
    // the last one to 2 kDepth - 1 steps: the slots in flight, the first ones refilled if needed
    const int rem = s1 - cs;
#pragma unroll
    for (int u = 0; u < kDepth; ++u)
      if (u < rem) {
        step(ring[u]);
        if (kDepth + u < rem) {
          load(ring[u], lc);
          __builtin_amdgcn_sched_barrier(0);
          advance();
        }
      }
#pragma unroll
    for (int u = 0; u + 1 < kDepth; ++u)
      if (kDepth + u < rem) step(ring[u]);
  }
  __syncthreads();
  // a tile begun in this wavefront's range and not finished there: its own sums and the others'
  const int tl = s1 > s0 ? (s1 - 1) / C : 0;
  if (s1 > s0 && s1 - tl * C < C && tl * C >= s0) emit(tl, 1, (tl + 1) * C);
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(aside) != 0, 0)) {
    // The outputs set aside of this wavefront's tiles: those of a row with an infinite scale (all of
    // the row's are), and those that are NaN in this order too.
    auto slices = [&](const uint8_t* wire, int row, int col, bool& inf) {
      const uint32_t blk = fastdiv((uint32_t)row, p.tdiv), in = row - blk * (uint32_t)p.tile_m;
      const uint8_t* q = wire + (size_t)blk * p.blk_bytes + (size_t)in * K;
      const uint16_t* sr =
          (const uint16_t*)(wire + (size_t)blk * p.blk_bytes + share.scales) + (size_t)in * ng;
      double sum = 0.0;
#pragma unroll 1
      for (int k = 0; k < K; k += 16) {
        double t = 0.0;
#pragma unroll 1
        for (int j = k; j < k + 16; ++j) {
          float x;
          if constexpr (XS == X_BF16) {
            x = bf16_to_f32(ld_global((const uint16_t*)p.x + (size_t)col * p.x_stride + j));
          } else if constexpr (XS == X_F32) {
            x = ld_global((const float*)p.x + (size_t)col * p.x_stride + j);
          } else {
            const float4* c = s_x + ((size_t)(j / kChunk) * nb + col) * kColUnits;
            x = ((const float*)(c + ((j >> 2) & 3) * 16 + j % kChunk / 16))[j & 3];
          }
          t = fma(sbyte(ld_global(q + j) ^ (p.xor_mask & 0xffu), 0), (double)x, t);
        }
        const float s = bf16_to_f32(ld_global(sr + (k >> p.gshift)));
        inf |= __builtin_isinf(s);
        sum = fma((double)s, t, sum);
      }
      return sum;
    };
    for (int tile = (s0 + C - 1) / C; tile * C < s1; ++tile) {
      for (int o = lane; o < TR * NB * 4; o += 64) {
        const int col = o / TR, row = (t0 + tile) * TR + o % TR;
        if (row >= p.M || col >= nb) continue;
        bool inf = false;
        const double v = slices(p.w, row, col, inf);
        const double v2 = DUAL ? slices(p.w2, row, col, inf) : v;
        if (inf || v != v || v2 != v2) store(row, col, v, v2);
      }
    }
  }
  if (p.epi != EPI_BF16_ARGMAX) return;
  __syncthreads();
  // one candidate per workgroup and batch row; an atomic only when it beats the published value
  if (tid < nb && s_best[tid]) {
    const unsigned long long cur =
        __hip_atomic_load(p.argmax + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (s_best[tid] > cur) atomicMax(p.argmax + tid, s_best[tid]);
  }
}

// Clocks of one wavefront step: 16 k positions of R NM weight rows (dequantizing fma) and their
// products with NB column groups, plus the x conversions and about 100 of loads and addresses.
int step_clocks(int nbg, int rows) { return 16 * (rows * (17 * nbg + 5) + 5 * nbg) + 100; }

// Steps of the busiest workgroup (the launch keeps them below 2^28).
long long max_steps(int M, int K, int rows) {
  const long long tiles = ((long long)M + rows - 1) / rows;
  return (tiles + kCUs - 1) / kCUs * ((K + kChunk - 1) / kChunk);
}

// Rows per tile / 4, 1, 2 or 4 up to `most` (and 3 with `three`): the smallest time of the busiest
// workgroup's wavefronts, ceil(steps / 8) steps.
int pick_rows(int M, int K, int nbg, int nm, int most, bool three) {
  int best = 0;
  long long cost = 0;
  for (int r = 1; r <= most; ++r) {
    if (r == 3 && !three) continue;
    const long long c =
        (max_steps(M, K, 4 * r) + kWaves - 1) / kWaves * step_clocks(nbg, r * nm);
    if (!best || c < cost || (c == cost && r > best)) {
      best = r;
      cost = c;
    }
  }
  return best;
}

// The launch of a kernel over the tiles of R NM * 4 rows, `groups` workgroups for each share.
template <class Kernel>
void enqueue(Kernel kernel, const GemvParams& p, int rows, int groups, size_t lds, hipStream_t s) {
  const long long tiles = ((long long)p.M + rows - 1) / rows;
  const unsigned grid = (unsigned)(tiles < kCUs ? tiles : kCUs);
  const Shares share = {(int)(tiles / grid), (int)(tiles % grid), (size_t)p.tile_m * p.K};
  hipLaunchKernelGGL(kernel, dim3(grid, groups), dim3(kThreads), lds, s, p, share);
}

// Matrices of so few tiles that every group of four batch rows has CUs of its own run one group per
// workgroup (bf16 x): with all groups in each, most CUs idle (us at K = 16384, M = 64, B = 5 / 15:
// 13.3 / 22.2 together, 10.9 / 10.9 apart; the kernel before this one 11.9 / 12.1).
bool launch_split(const GemvParams& p, hipStream_t s) {
  const int groups = (p.nb + 3) / 4;
  if (p.pro != PRO_BF16 || groups < 2 || ((long long)p.M + 3) / 4 * groups > kCUs) return false;
  if (p.gshift == 4)
    enqueue(gemv_rows_kernel<1, 1, false, X_BF16, true, 1, true>, p, 4, groups, 0, s);
  else
    enqueue(gemv_rows_kernel<1, 1, false, X_BF16, false, 1, true>, p, 4, groups, 0, s);
  return true;
}

template <int NB, int R, bool DUAL, int XS>
void launch(const GemvParams& p, size_t lds, hipStream_t s) {
  auto go = [&](auto g16, auto dep) {
    enqueue(gemv_rows_kernel<NB, R, DUAL, XS, decltype(g16)::value, decltype(dep)::value>, p, 4 * R,
            1, lds, s);
  };
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  if constexpr (R <= 2) {  // groups of 16 run at these tile heights
    if (p.gshift == 4) return go(std::true_type(), One());
  }
  // One step in flight per wavefront, the others' compute hiding its loads: a deeper ring measured
  // slower (us at depth 1 / 2 / 3: 4096 x 12288 B = 4 17.9 / 18.9 / 20.0, gate/up of 4B 22.8 / 22.9 /
  // 24.2) except over many steps (the 151936 x 1024 head, 19 a wavefront: 52.2 / 48.8 / 49.2; the line
  // lies between its 19 and the 6 of 4096 x 12288).
  if constexpr (R == 4 && NB <= 2 && !DUAL && XS != X_F32) {
    if (max_steps(p.M, p.K, 4 * R) >= 12 * kWaves) return go(std::false_type(), Two());
  }
  go(std::false_type(), One());
}

template <int NB, int XS>
void launch_rows(const GemvParams& p, size_t lds, hipStream_t s) {
  const int R = pick_rows(p.M, p.K, NB, 1, p.gshift == 4 ? 2 : 4, NB == 1);
  if constexpr (NB == 1) {
    if (R == 3) return launch<NB, 3, false, XS>(p, lds, s);
  }
  if (R == 1) launch<NB, 1, false, XS>(p, lds, s);
  else if (R == 2) launch<NB, 2, false, XS>(p, lds, s);
  else launch<NB, 4, false, XS>(p, lds, s);
}

template <int NB>
void launch_nb(const GemvParams& p, bool dual, size_t lds, hipStream_t s) {
  const bool staged = p.pro == PRO_RMS_BF16 || p.pro == PRO_RES_RMS_F32;
  if (dual) {
    if (pick_rows(p.M, p.K, NB, 2, 2, false) == 1)
      launch<NB, 1, true, X_LDS>(p, lds, s);
    else
      launch<NB, 2, true, X_LDS>(p, lds, s);
  } else if (staged) {
    launch_rows<NB, X_LDS>(p, lds, s);
  } else if (p.pro == PRO_F32) {
    if constexpr (NB <= 2) launch_rows<NB, X_F32>(p, lds, s);  // launched up to eight rows at a time
  } else {
    launch_rows<NB, X_BF16>(p, lds, s);
  }
}

}  // namespace

namespace iron {

// Whether the staged columns of a call's B rows of K elements fit the LDS, beside the static LDS of
// the largest tile (R NM = 4): s_part and the steps' weights and scales.
bool gemv_rows_fits(int B, int K) {
  const size_t col = (size_t)((K + kChunk - 1) / kChunk) * kColUnits * 16;
  const int fixed = kWaves * (2 * ((B + 3) / 4) * 4 * 16 * 8 + 4096 + 16 + 1024);
  return col * B + fixed <= (size_t)kMaxLds;
}

int gemv_rows_launch(const GemvParams& p, int B, bool dual, hipStream_t stream, const char* fn) {
  if (max_steps(p.M, p.K, 4) >= (1ll << 28))
    return fail(IRON_ERR_SHAPE, "%s: M=%d K=%d too large", fn, p.M, p.K);
  const bool staged = p.pro == PRO_RMS_BF16 || p.pro == PRO_RES_RMS_F32;
  const size_t col = (size_t)((p.K + kChunk - 1) / kChunk) * kColUnits * 16;
  // batch rows per launch: all of them, or as many as the staged columns leave room for
  int per = p.pro == PRO_F32 && B > 8 ? 8 : B;
  if (staged) {
    while (per > 1 && !gemv_rows_fits(per, p.K)) --per;
    if (!gemv_rows_fits(per, p.K))
      return fail(IRON_ERR_UNSUPPORTED, "%s: K=%d exceeds the LDS-staged GEMV limit", fn, p.K);
  }
  for (int b0 = 0; b0 < B; b0 += per) {
    const int n = B - b0 < per ? B - b0 : per;
    const GemvParams q = rows_of(p, b0, n);
    const size_t lds = staged ? col * n : 0;
    if (!launch_split(q, stream)) switch ((n + 3) / 4) {
      case 1: launch_nb<1>(q, dual, lds, stream); break;
      case 2: launch_nb<2>(q, dual, lds, stream); break;
      case 3: launch_nb<3>(q, dual, lds, stream); break;
      default: launch_nb<4>(q, dual, lds, stream); break;
    }
    const int st = check_launch(fn);
    if (st) return st;
  }
  return IRON_OK;
}

}  // namespace iron
