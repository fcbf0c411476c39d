// The decoder's matrix products in a decode step: out = x W^T for up to 64
// rows of x, with the SiLU-and-multiply of a gated MLP in the epilogue on
// request.
//
// Reference: the engine's linear layers (linear.py: F.linear; the MLP's
// activation.py:16-19), which a decode step calls with one row per sequence.
// Operands are bf16, products and sums fp32 (v_mfma_f32_16x16x32_bf16),
// rounded once.
//
// With so few rows a product is one pass over its weights (8 MB, the q/k/v of
// a 1024-wide layer, are 1.3 us at 6.4 TB/s) and what costs is the latency
// around it and the reads of x by every CU.  So k is shared out over the
// waves of a workgroup until a wave's share is one memory round trip, and
// there are about as many workgroups as CUs.  60 rows, weights not in cache,
// us a product, before (the library's products, the gated one with
// mkv_silu_mul behind it) and now: 4096 x 1024 11.2 / 6.3, 1024 x 2048 9.7 /
// 5.3, 1024 x 3072 12.0 / 7.5, 2 x 3072 x 1024 gated 14.7 / 9.3, 151936 x 1024
// 85 / 76; one row: 7.5 / 4.5, 8.7 / 5.0, 11.9 / 6.6, 10.4 / 5.6.  With the
// residual added 1024 x 2048 takes 5.4 and 1024 x 3072 7.7; normalised (before:
// behind mkv_rmsnorm with its residual addition) 4096 x 1024 15.1 / 9.6 and the
// gated one 18.5 / 11.2, one row 10.8 / 5.4 and 13.7 / 6.8: those are the forms
// of a decoder layer.
//
// The MFMA's rows are 16 output features (A = W, straight from memory: the
// loads of two k-steps cover 16 whole lines), its columns 16 rows of x, so a
// lane ends with 4 consecutive features of one row.
#include "mkv_device.hpp"

namespace mkv {
namespace {

constexpr int kLinMaxRows = 64;
constexpr int kNormMaxK = 2048;  // mkv_rmsnorm's
constexpr int64_t kLinMaxStride = (int64_t)1 << 20;  // x's offsets are 32 bits
constexpr int kCus = 256;
constexpr int kXcds = 8;
constexpr size_t kLdsPerCu = 160 * 1024;

struct LinearArgs {
  uint16_t* out;      // (rows, n)
  const uint16_t* x;  // (rows, k), row stride x_stride
  const uint16_t* w;  // (n, k), with act: (2 n, k), gate rows then up rows
  int64_t x_stride;
  int rows, n, k;
  int m_groups;       // groups of 16 MT rows
  const uint16_t* norm;      // NORM: RMSNorm weight (k)
  float eps;
  const uint16_t* residual;  // (rows, n) added to the rounded product, or null; may be out
};

MKV_DEV bf16x8 ld_op(const uint16_t* p) { return __builtin_bit_cast(bf16x8, ld16(p)); }

MKV_DEV uint2 pack_bf16x4(const float* x) {
  return make_uint2(f32_to_bf16_bits(x[0]) | (f32_to_bf16_bits(x[1]) << 16),
                    f32_to_bf16_bits(x[2]) | (f32_to_bf16_bits(x[3]) << 16));
}

// Element offset of k-step u from a lane's first (16 kg): the lane's 8
// elements of two successive steps are 32 bytes together, so both steps' loads
// touch the same 16 whole lines (the order within k is free).
MKV_DEV constexpr int step_off(int u) { return 64 * (u >> 1) + 8 * (u & 1); }

// Workgroup barrier that leaves loads in flight alone: this wave's LDS
// accesses are done.
MKV_DEV void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// ---------------------------------------------------------------------------
// Split form: a workgroup owns 16 features (with ACT: 16 gate and the 16 up
// features of the same outputs) and MT tiles of 16 rows, its waves share out
// k, and their sums are joined in LDS (in wave order: the result does not
// depend on timing).  A wave issues BLK k-steps' loads at once, so that a
// product whose k is 32 BLK x waves is a single memory round trip.  x comes by
// LDS DMA, whole lines an instruction: read as MFMA operands straight from
// memory (16 half lines an instruction, the same ones by every CU) it took
// 7.5 us for 4096 x 1024 at 60 rows, not 6.2.
// ---------------------------------------------------------------------------
//
// NORM (products of one round trip): x's rows are RMS-normalised on the way,
// round(x * (1 / rms) * weight) as mkv_rmsnorm rounds it.  Every workgroup
// works the rows' sums of squares out of the x it reads anyway, its waves'
// parts joined in LDS ahead of the product.  At 60 rows the two norms of a
// layer took 5 us each as launches of their own (add, norm, one row a wave);
// with them and the residual additions here a decode step of 8 layers went
// from 580 to 556 us.
template <int MT, int BLK, bool ACT, bool NORM>
__global__ __launch_bounds__(1024) void linear_split_kernel(LinearArgs a) {
  constexpr int NT = ACT ? 2 : 1;
  extern __shared__ __align__(16) char smem[];
  f32x4* part = reinterpret_cast<f32x4*>(smem);  // [wave][NT][MT][lane]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int waves = blockDim.x >> 6;
  const int c = lane & 15, kg = lane >> 4;
  // consecutive workgroups (the row groups of one feature tile) on one XCD
  const int nwg = gridDim.x;
  const int b = nwg % kXcds == 0 ? (blockIdx.x % kXcds) * (nwg / kXcds) + blockIdx.x / kXcds : blockIdx.x;
  const int n0 = (b / a.m_groups) * 16, m0 = (b % a.m_groups) * 16 * MT;

  const int steps = a.k / 32 / waves;
  const int kw = wave * steps * 32;
  const uint16_t* wp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) wp[t] = a.w + (int64_t)(n0 + t * a.n + c) * a.k + kw + 16 * kg;
  // x by LDS DMA: BLK steps are kCh 16-byte chunks of each of 16 MT rows, slot
  // i of the wave's part holding chunk (i % kCh) ^ swz of row i / kCh, so that
  // a load instruction covers whole lines and the 16 rows of an operand read
  // hit 16 positions of 256 bytes
  constexpr int kCh = 4 * BLK, kRowsX = 16 * MT, kDmas = kRowsX * kCh / 64;
  auto swz = [](int row) { return kCh % 16 == 0 ? row & 15 : (row >> 1) & 7; };
  char* xs = smem + wave * (kRowsX * kCh * 16);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      (void*)a.x, (short)0, (int)(2 * ((a.rows - 1) * (int)a.x_stride + a.k)), 0x00020000);
  uint32_t x_off[kDmas];
#pragma unroll
  for (int d = 0; d < kDmas; ++d) {
    const int i = 64 * d + lane, row = i / kCh, ch = (i % kCh) ^ swz(row);
    x_off[d] = 2u * (uint32_t)(min(m0 + row, a.rows - 1) * (int)a.x_stride + kw + 8 * ch);
  }

  f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < steps; s += BLK) {
    bf16x8 wf[BLK][NT], nf[NORM ? BLK : 1];
#pragma unroll
    for (int d = 0; d < kDmas; ++d)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (__attribute__((address_space(3))) void*)(xs + 1024 * d), 16,
                                               (int)x_off[d], 64 * s, 0, 0);
#pragma unroll
    for (int u = 0; u < BLK; ++u)
#pragma unroll
      for (int t = 0; t < NT; ++t) wf[u][t] = ld_op(wp[t] + 32 * s + step_off(u));
    if constexpr (NORM) {
#pragma unroll
      for (int u = 0; u < BLK; ++u) nf[u] = ld_op(a.norm + kw + 16 * kg + 32 * s + step_off(u));
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): x has landed (the wave's own: no barrier)
    asm volatile("" ::: "memory");
    auto x_op = [&](int u, int j) {  // chunk of elements step_off(u) + 16 kg of row 16 j + c
      const int row = 16 * j + c, ch = (8 * (u >> 1) + (u & 1) + 2 * kg) ^ swz(row);
      return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(xs + (row * kCh + ch) * 16));
    };
    float inv[MT];
    if constexpr (NORM) {
      float* sq = reinterpret_cast<float*>(smem + waves * (kRowsX * kCh * 16));  // [MT][16][wave]
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        float ss = 0.0f;
#pragma unroll
        for (int u = 0; u < BLK; ++u) {
          const bf16x8 xf = x_op(u, j);
#pragma unroll
          for (int e = 0; e < 8; e += 2) {
            const bf16x2 p = {xf[e], xf[e + 1]};
            ss = __builtin_amdgcn_fdot2_f32_bf16(p, p, ss, false);
          }
        }
        ss += __shfl_xor(ss, 16);
        ss += __shfl_xor(ss, 32);
        if (kg == 0) sq[(16 * j + c) * waves + wave] = ss;
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        float ss = 0.0f;
        for (int w = 0; w < waves; w += 4) {
          const f32x4 q = *reinterpret_cast<const f32x4*>(sq + (16 * j + c) * waves + w);
          ss += (q[0] + q[1]) + (q[2] + q[3]);
        }
        inv[j] = 1.0f / __builtin_sqrtf(ss / (float)a.k + a.eps);
      }
    }
#pragma unroll
    for (int u = 0; u < BLK; ++u)
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        bf16x8 xf = x_op(u, j);
        if constexpr (NORM) {
#pragma unroll
          for (int e = 0; e < 8; ++e) xf[e] = (__bf16)((float)xf[e] * inv[j] * (float)nf[u][e]);
        }
#pragma unroll
        for (int i = 0; i < NT; ++i)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][i], xf, acc[i][j], 0, 0, 0);
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  __syncthreads();  // the sums take the place of x
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) part[((wave * NT + i) * MT + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  for (int j = wave; j < MT; j += waves) {
    f32x4 sum[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) sum[i] = part[(i * MT + j) * 64 + lane];
#pragma unroll 4
    for (int w = 1; w < waves; ++w)
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const f32x4 p = part[((w * NT + i) * MT + j) * 64 + lane];
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[i][r] += p[r];
      }
    const int m = m0 + 16 * j + c;
    if (m >= a.rows) continue;
    const int64_t o = (int64_t)m * a.n + n0 + 4 * kg;
    uint2 res = make_uint2(0, 0);
    if (!ACT && a.residual) res = *reinterpret_cast<const uint2*>(a.residual + o);
    float y[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (ACT) {  // on gate and up rounded to bf16, as mkv_silu_mul reads them
        const float g = bf16_bits_to_f32(f32_to_bf16_bits(sum[0][r]));
        const float u = bf16_bits_to_f32(f32_to_bf16_bits(sum[NT - 1][r]));
        y[r] = g / (1.0f + __expf(-g)) * u;
      } else {
        y[r] = sum[0][r];
        if (a.residual)  // the product rounded first, as a product of its own
          y[r] = bf16_bits_to_f32(f32_to_bf16_bits(y[r])) +
                 bf16_bits_to_f32(((r < 2 ? res.x : res.y) >> (16 * (r & 1))) & 0xffffu);
      }
    }
    *reinterpret_cast<uint2*>(a.out + o) = pack_bf16x4(y);
  }
}

// ---------------------------------------------------------------------------
// Streaming form, for products with many more feature tiles than CUs (an LM
// head): one 8-wave workgroup a CU takes a contiguous range of feature tiles.
// Each wave keeps its eighth of x (STEPS k-steps of every row) in registers and
// streams its eighth of the tiles' weights through a ring of three groups of
// tiles (pairs, single ones past k 1024), two groups (128 KB a CU for k 1024 and
// 2048) in flight ahead of the one it multiplies; the waves' sums of a group meet
// in LDS (double-buffered, one barrier a group that leaves the loads in flight),
// where wave w joins tile w / 4, rows 16 (w % 4).
// 151936 x 1024 (311 MB of weights): 63 us for one row, 78 for 60 (the writes of
// 18 MB of logits); plain loads, since non-temporal ones took 68 and 88.
// ---------------------------------------------------------------------------
constexpr int kStreamWaves = 8;

template <int MT, int STEPS>
__global__ __launch_bounds__(kStreamWaves* kWave) __attribute__((amdgpu_waves_per_eu(2))) void linear_stream_kernel(
    LinearArgs a) {
  static_assert(STEPS % 2 == 0, "step_off goes by pairs of k-steps");
  constexpr int kK = 32 * STEPS * kStreamWaves;
  constexpr int TP = STEPS <= 4 ? 2 : 1;  // tiles of a group
  extern __shared__ __align__(16) char smem[];
  f32x4* part = reinterpret_cast<f32x4*>(smem);  // [2][wave][tile][MT][lane]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, kg = lane >> 4;
  const int tiles = a.n / 16;
  const int nwg = gridDim.x;
  const int b = nwg % kXcds == 0 ? (blockIdx.x % kXcds) * (nwg / kXcds) + blockIdx.x / kXcds : blockIdx.x;
  const int t0 = (int)((int64_t)tiles * b / nwg), t1 = (int)((int64_t)tiles * (b + 1) / nwg);
  const int groups = (t1 - t0 + TP - 1) / TP;
  if (groups == 0) return;

  const int k0 = wave * 32 * STEPS + 16 * kg;
  const __amdgpu_buffer_rsrc_t wr =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.w, (short)0, (int)(2u * (uint32_t)a.n * kK), 0x00020000);
  const int w_off = 2 * (c * kK + k0);
  // (past the last tile: its weights again, so that every path issues the same
  // loads and the waits count them exactly)
  auto load_group = [&](int p, bf16x8 (&f)[TP][STEPS]) {
#pragma unroll
    for (int i = 0; i < TP; ++i) {
      const int tile_off = (int)(min(t0 + TP * p + i, t1 - 1) * (2u * 16 * kK));
#pragma unroll
      for (int u = 0; u < STEPS; ++u)
        f[i][u] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(wr, w_off + 2 * step_off(u), tile_off, 0));
    }
  };
  bf16x8 f0[TP][STEPS], f1[TP][STEPS], f2[TP][STEPS], xf[MT][STEPS];
  load_group(0, f0);
#pragma unroll
  for (int j = 0; j < MT; ++j)
#pragma unroll
    for (int u = 0; u < STEPS; ++u)
      xf[j][u] = ld_op(a.x + (int64_t)min(16 * j + c, a.rows - 1) * a.x_stride + k0 + step_off(u));
  load_group(1, f1);

  const __amdgpu_buffer_rsrc_t out =
      __builtin_amdgcn_make_buffer_rsrc(a.out, (short)0, (int)(2u * (uint32_t)a.rows * (uint32_t)a.n), 0x00020000);
  const int red_tile = wave >> 2, red_m = 16 * (wave & 3) + c;
  auto step = [&](int p, bf16x8 (&cur)[TP][STEPS], bf16x8 (&ahead)[TP][STEPS]) {
    load_group(p + 2, ahead);
    __builtin_amdgcn_sched_barrier(0);
    f32x4* buf = part + (p & 1) * (kStreamWaves * TP * MT * 64);
#pragma unroll
    for (int i = 0; i < TP; ++i) {
      f32x4 acc[MT];
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < STEPS; ++u)
#pragma unroll
        for (int j = 0; j < MT; ++j)
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cur[i][u], xf[j][u], acc[j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < MT; ++j) buf[((wave * TP + i) * MT + j) * 64 + lane] = acc[j];
    }
    lds_barrier();
    if (TP == 1 && red_tile) return;  // (a single tile: its rows are the first four waves')
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kStreamWaves; ++w) {
      const f32x4 q = buf[((w * TP + red_tile) * MT + min(wave & 3, MT - 1)) * 64 + lane];
#pragma unroll
      for (int r = 0; r < 4; ++r) sum[r] += q[r];
    }
    const float y[4] = {sum[0], sum[1], sum[2], sum[3]};
    const uint2 o = pack_bf16x4(y);
    const int tile = t0 + TP * p + red_tile;
    const bool ok = red_m < a.rows && tile < t1;
    const uint32_t off = ok ? 2u * ((uint32_t)red_m * (uint32_t)a.n + (uint32_t)(tile * 16 + 4 * kg)) : 0xfffffff8u;
    __builtin_amdgcn_raw_buffer_store_b64(u32x2{o.x, o.y}, out, (int)off, 0, 0);
  };
  for (int p = 0;;) {
    step(p, f0, f2);
    if (++p >= groups) break;
    step(p, f1, f0);
    if (++p >= groups) break;
    step(p, f2, f1);
    if (++p >= groups) break;
  }
}

// How a product runs; kind 0: not at all (the caller's own product).
struct LinearPlan {
  int kind;  // 1 split, 2 streaming
  int mt, waves, blk;
};

// LDS of a split workgroup: x's parts (normalised: and the waves' sums of
// squares), then the waves' sums in their place.
size_t split_lds(const LinearPlan& p, int act, int norm) {
  const size_t sums = (size_t)p.waves * (act ? 2 : 1) * p.mt * 1024;
  const size_t x = (size_t)p.waves * p.mt * (16 * p.blk * 64 + (norm ? 64 : 0));
  return sums > x ? sums : x;
}

LinearPlan plan_linear(int64_t rows, int n, int k, int act, int norm) {
  LinearPlan p{0, 0, 0, 0};
  if (rows < 1 || rows > kLinMaxRows || n < 16 || n % 16 || k < 32 || k % 32) return p;
  if (norm && k > kNormMaxK) return p;
  const int m_tiles = (int)(rows + 15) / 16, n_tiles = n / 16;
  // Streaming, for more than 16 rows (at most 16 are as fast or faster in the
  // library: 151936 x 1024 one row 62 us and 63 here, 16 rows 65 / 69), of k up
  // to what a wave holds of x and offsets of 32 bits, from 16 feature tiles a CU
  // on (8 at k 512): with fewer, a range's whole groups weigh too much (40 rows,
  // 50272 features: k 1024 22.4 us and 27.3 here, 1536 33.6 / 35.8).  From there
  // on the library goes from a little faster to half as fast, with its own
  // tiling: 40 rows, k 512 / 1024 / 1536 / 2048: 79984 features 42.2 / 58.7 / 83.0
  // / 80.1 and 20.3 / 39.3 / 54.6 / 72.7 here, 115200 32.1 / 52.7 / 86.1 / 102.9
  // and 28.3 / 56.1 / 76.7 / 101.7, 128256 41.1 / 57.3 / 101.4 / 123.6 and 31.2 /
  // 59.1 / 86.3 / 110.0, 200064 102.4 / 144.0 / 200.9 / 195.1 and 47.0 / 90.4 /
  // 134.7 / 167.3, 256000 61.7 / 111.8 / 171.5 / 233.7 and 58.7 / 114.2 / 168.8 /
  // 212.4.
  if (!act && n_tiles >= 8 * kCus) {
    if (norm || k % 512 || k > 2048 || m_tiles < 2 || n_tiles < (k == 512 ? 8 : 16) * kCus ||
        (int64_t)k * n * 2 >= ((int64_t)1 << 31))
      return p;
    p.kind = 2;
    p.mt = m_tiles;
    p.blk = k / 256;
    return p;
  }
  // Split up to 2^20 (feature tiles x row tiles x k: 32 MB of x read by the
  // workgroups) and k 4096; past either the library is as fast or faster.
  // 64 rows: 4096 x 1024 11.6 us and 7.7 here, 2048 x 2048 11.9 / 7.2, 6144 x
  // 1024 11.9 / 12.2, 4096 x 4096 15.4 / 21.0; 16 rows: 4096 x 4096 15.9 /
  // 11.2, 6144 x 4096 16.0 / 17.2, 2048 x 6144 12.2 / 13.1.
  if ((int64_t)n_tiles * m_tiles * k > (1 << 20) || k > 4096) return p;
  // Waves: as many as leave each of them one or two times 4 or 6 k-steps
  // (2560 = 4 waves x 5 times 4 at 32 rows: 9.5 us and 10.5 here).
  const int steps = k / 32;
  for (int waves : {16, 8, 4}) {
    if (steps % waves) continue;
    const int per = steps / waves;
    if (waves == 16 && per < 4) continue;
    const int blk = per % 4 == 0 ? 4 : (per % 6 == 0 ? 6 : 0);
    if (!blk || per > (norm ? 1 : 2) * blk) continue;
    p.waves = waves;
    p.blk = blk;
    break;
  }
  if (!p.blk) return p;
  p.kind = 1;
  // Rows a workgroup: all of them (the weights are read once) where that still
  // makes a workgroup a CU, else fewer: 1024 features are 64 tiles, 256
  // workgroups at 16 rows each.
  for (p.mt = m_tiles > 2 ? 4 : m_tiles; p.mt > 1 && (int64_t)n_tiles * ((m_tiles + p.mt - 1) / p.mt) < kCus;) p.mt /= 2;
  if (act && p.mt == 4) p.mt = 2;
  if ((p.waves == 16 || p.blk == 6) && p.mt == 4) p.mt = 2;
  if (act && norm && p.blk == 6) p.mt = 1;  // (two row tiles do not fit the registers)
  // Not where one workgroup fills a CU's LDS and there are more of them than
  // CUs: the few of the second round take as long as all of the first.  Here and
  // in the library, us: 2560 x 1536 at 48 rows 10.4 and 9.5, 1536 x 3072 at 48
  // 13.3 / 10.2 and gated 19.9 / 13.7, normalised 2560 x 2048 at 33 19.8 / 15.6 and
  // 4608 x 1024 at 33 17.2 / 15.1; but plain 4608 x 1024 at 33 10.4 / 11.8.
  // Two a CU hide each other, in more rounds too: 3072 x 2048 at 32 rows 8.8 /
  // 11.5, 24576 x 512 at 16 8.7 / 12.6, 8192 x 2048 normalised at 16 16.1 / 18.4.
  const int64_t wgs = (int64_t)n_tiles * ((m_tiles + p.mt - 1) / p.mt);
  if (wgs > kCus && 2 * split_lds(p, act, norm) > kLdsPerCu && (k > 1024 || norm)) return LinearPlan{0, 0, 0, 0};
  return p;
}

template <int MT, bool ACT, bool NORM>
void launch_split(const LinearArgs& a, const LinearPlan& p, hipStream_t s) {
  const dim3 grid((unsigned)(a.n / 16 * a.m_groups)), block(p.waves * kWave);
  const size_t lds = split_lds(p, ACT, NORM);
  constexpr bool kFour = MT == 4 || (MT == 2 && ACT && NORM);  // plan_linear's
  if (kFour || p.blk == 4)
    hipLaunchKernelGGL((linear_split_kernel<MT, 4, ACT, NORM>), grid, block, lds, s, a);
  else
    hipLaunchKernelGGL((linear_split_kernel<MT, kFour ? 4 : 6, ACT, NORM>), grid, block, lds, s, a);
}

template <bool ACT, bool NORM>
void launch_rows(const LinearArgs& a, const LinearPlan& p, hipStream_t s) {
  if constexpr (!ACT) {
    if (p.mt == 4) return launch_split<4, false, NORM>(a, p, s);
  }
  if (p.mt == 2) launch_split<2, ACT, NORM>(a, p, s);
  else launch_split<1, ACT, NORM>(a, p, s);
}

template <int STEPS>
void launch_stream(const LinearArgs& a, int mt, hipStream_t s) {
  const dim3 grid(kCus), block(kStreamWaves * kWave);
  const size_t lds = (size_t)2 * kStreamWaves * (STEPS <= 4 ? 2 : 1) * mt * 64 * sizeof(f32x4);
  switch (mt) {
    case 2: hipLaunchKernelGGL((linear_stream_kernel<2, STEPS>), grid, block, lds, s, a); break;
    case 3: hipLaunchKernelGGL((linear_stream_kernel<3, STEPS>), grid, block, lds, s, a); break;
    default: hipLaunchKernelGGL((linear_stream_kernel<4, STEPS>), grid, block, lds, s, a); break;
  }
}

}  // namespace
}  // namespace mkv

using namespace mkv;

extern "C" int mkv_linear_supported(int64_t rows, int n, int k, int act, int norm, int dtype) {
  return dtype == MKV_DTYPE_BF16 && plan_linear(rows, n, k, act, norm).kind != 0;
}

extern "C" int mkv_linear(void* out, const void* x, int64_t x_row_stride, const void* w,
                          const void* norm_weight, float eps, const void* residual, int64_t rows, int n, int k,
                          int act, int dtype, void* stream) {
  if (dtype != MKV_DTYPE_BF16) return MKV_ERR_UNSUPPORTED_DTYPE;
  const LinearPlan p = plan_linear(rows, n, k, act, norm_weight != nullptr);
  if (!p.kind || x_row_stride < k || x_row_stride > kLinMaxStride) return MKV_ERR_BAD_SHAPE;
  if (residual && (act || p.kind == 2)) return MKV_ERR_BAD_SHAPE;
  if (!out || !x || !w) return MKV_ERR_NULL_POINTER;
  if (((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) |
        reinterpret_cast<uintptr_t>(norm_weight) | reinterpret_cast<uintptr_t>(residual)) & 15u) ||
      x_row_stride % 8)
    return MKV_ERR_MISALIGNED;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  LinearArgs a{reinterpret_cast<uint16_t*>(out), reinterpret_cast<const uint16_t*>(x),
               reinterpret_cast<const uint16_t*>(w), x_row_stride, (int)rows, n, k, 1,
               reinterpret_cast<const uint16_t*>(norm_weight), eps, reinterpret_cast<const uint16_t*>(residual)};
  const int m_tiles = (int)(rows + 15) / 16;
  if (p.kind == 2) {
    switch (p.blk) {
      case 2: launch_stream<2>(a, p.mt, s); break;
      case 4: launch_stream<4>(a, p.mt, s); break;
      case 6: launch_stream<6>(a, p.mt, s); break;
      default: launch_stream<8>(a, p.mt, s); break;
    }
  } else {
    a.m_groups = (m_tiles + p.mt - 1) / p.mt;
    if (act) {
      if (norm_weight) launch_rows<true, true>(a, p, s);
      else launch_rows<true, false>(a, p, s);
    } else {
      if (norm_weight) launch_rows<false, true>(a, p, s);
      else launch_rows<false, false>(a, p, s);
    }
  }
  return (int)hipGetLastError();
}
