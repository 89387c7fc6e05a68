// Weight gradient of a linear layer (gfx950): dW[n][k] = sum_m dY[m][n] X[m][k] over M tokens, the autograd of
// the projections at transformer.py:208-213, :263, :300 and of the loss's logits (:96-98) with respect to their weights.
// bf16 operands as the forward and backward leave them (token rows), fp32 sums, fp32 or bf16 dW.
//
// What bounds it: MFMA, with the LDS reads close behind.  The reduction runs over tokens, the rows of both operands, so
// both fragments come from transpose reads (ds_read_b64_tr_b16, 128 bytes a clock per CU, half of a plain 16-byte read):
// a wave of 128 (n) x 64 (k) reads 6 KiB per 16 tokens for 8 MFMAs (32x32x16), 384 clocks of the CU's LDS for eight
// waves against 512 clocks of MFMA, and the tiles' arrival takes another 128.  A 256 x 256 tile asks L2 for 32 bytes a
// clock per CU; a 128 x 128 one would ask for 64, all that the CU's memory pipe moves.
//
// Tokens arrive in stages of 32 by direct-to-LDS loads into a 4-stage ring.  A stage's rows keep their order, chunk c
// of 16 bytes at position c ^ 4 (row mod 4), so the four rows of a half-wave's transpose read fall on four different
// 64-byte bank groups.  The one barrier of a stage lies between its two 16-token halves: the first half's products run
// under the second half's reads, and the next stage's first reads under the second half's products.
//
// Few weights have as many 256 x 256 tiles as the chip has CUs, so the tokens are cut into S segments and a second
// kernel adds the segments' fp32 partials in order (no atomics: the result is bitwise reproducible).  S and the tile
// come from a cost model (wg_plan in plans.h).
//
// Measured (kernel trace of 40 calls, medians, main + segment sum with bf16 dW, against the library's product over the same
// operands in the same run; us):
//   M = 12288, N x K = 2560 x 1792: 105.2 + 10.8 (main 1072 TFLOP/s) against 218.7;  1792 x 1792: 72.1 + 12.0 against 121.3
//   1792 x 384: 23.1 + 7.1 against 73.1;  896 x 384: 17.0 + 6.2 against 70.6
//   M = 3001, 2048 x 2048: 29.7 + 9.3 against 44.5;  2048 x 512: 16.5 + 7.4 against 29.7
//   M = 8192, 4096 x 2048 (a chunk of the loss): 110.6 + 16.4 against 133.4; M = 3000, 4096 x 1792: 49.2 against 60.1
// In a training pass of one block (default dims, B = 6, T = 2048) the wide tile runs at 1060 TFLOP/s with MfmaUtil 46.9 %,
// the narrow one at 671 with 24.3 % (profiles/train_B6_T2048_default.txt); the pass went from 1897 to 1495 us.
#include <algorithm>

#include "mla_common.h"

namespace mla {

typedef short s16x4w __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4w lds_s16x4w;

struct WgParams {
  const bf16* dy;  // [M][N], row stride ldy
  const bf16* x;   // [M][K], row stride ldx
  void* out;       // [N][K], row stride ldo, fp32 or bf16
  float* part;     // S > 1: [segment][tile][wave][block][register quad][lane] quads of fp32
  int M, N, K;
  int64_t ldy, ldx, ldo;
  int S, seg;      // token segments, tokens per segment (a multiple of kWgSt)
  int nt, kt;      // tiles along n and k
  int out_f32;
};

constexpr int kWgRing = 4;    // stages
constexpr int kWgWaves = 8;

// TN x TK outputs per workgroup; WN waves along n, 8 / WN along k
template <int TN_, int TK_, int WN_>
struct WgCfg {
  static constexpr int TN = TN_, TK = TK_, WN = WN_, WK = kWgWaves / WN_;
  static constexpr int NB = TN / WN / 32, KB = TK / WK / 32;  // 32 x 32 blocks per wave
  static constexpr int YB = TN * 2, XB = TK * 2;              // bytes per staged row
  static constexpr int XOFF = kWgSt * YB;
  static constexpr int STAGE = kWgSt * (YB + XB);
  static constexpr int LOADS = STAGE / 1024 / kWgWaves;
  static constexpr int YL = XOFF / 1024;                      // the stage's first YL loads are dY's
  static_assert(STAGE % (1024 * kWgWaves) == 0 && YL % kWgWaves == 0 && kWgRing * STAGE <= 160 * 1024, "the ring fits the LDS");
};

template <int N>
__device__ __forceinline__ void wg_wait_vmem() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// block and quad of the accumulators -> the partial's place, and back in wgrad_reduce_kernel
template <class C>
__global__ __launch_bounds__(64 * kWgWaves, 1) void wgrad_kernel(WgParams p) {
  __shared__ __attribute__((aligned(1024))) unsigned char wg_lds[kWgRing * C::STAGE];
  // consecutive logical ids run on one XCD (hardware places id on XCD id % 8): tiles of one segment, which share
  // their token rows in that XCD's L2
  const int n_wg = gridDim.x;
  int id = blockIdx.x;
  if ((n_wg & 7) == 0) {
    id = (id & 7) * (n_wg >> 3) + (id >> 3);
  } else {
    const int q = n_wg >> 3, r = n_wg & 7, xcd = id & 7;
    id = xcd * q + min(xcd, r) + (id >> 3);
  }
  const int tiles = p.nt * p.kt;
  const int sg = id / tiles, tile = id - sg * tiles;
  const int tn = tile % p.nt, tk = tile / p.nt;
  const int n0 = tn * C::TN, k0 = tk * C::TK;
  const int m0 = sg * p.seg, rows = min(p.seg, p.M - m0);  // rows >= 1 (the host's S covers M exactly)
  const int n_st = (rows + kWgSt - 1) / kWgSt;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = w % C::WN, wk = w / C::WN;

  // the descriptors cover this segment's rows of the operand from column n0 (k0) on; lanes past them load nothing
  const buf_rsrc ry = make_rsrc(p.dy + (int64_t)m0 * p.ldy + n0, rows_bytes(rows, p.ldy, (p.N - n0) * 2));
  const buf_rsrc rx = make_rsrc(p.x + (int64_t)m0 * p.ldx + k0, rows_bytes(rows, p.ldx, (p.K - k0) * 2));
  const uint32_t lds0 = lds_addr(wg_lds);
  uint32_t voff[C::LOADS];  // this lane's bytes in each of the wave's loads, at the segment's first stage
#pragma unroll
  for (int j = 0; j < C::LOADS; ++j) {
    const int i = w + kWgWaves * j;  // load i of the stage: 1 KiB of staged rows
    const bool isy = kWgWaves * j < C::YL;  // (the same for every wave)
    const int rb = isy ? C::YB : C::XB;
    const int at = (isy ? i : i - C::YL) * 1024 + lane * 16;
    const int row = at / rb, pos = (at % rb) >> 4;
    voff[j] = (uint32_t)((int64_t)row * (isy ? p.ldy : p.ldx) * 2) + (uint32_t)((pos ^ (4 * (row & 3))) * 16);
  }
  const uint32_t ystep = (uint32_t)(kWgSt * p.ldy * 2), xstep = (uint32_t)(kWgSt * p.ldx * 2);
  auto issue = [&](int s, int slot) {
#pragma unroll
    for (int j = 0; j < C::LOADS; ++j) {
      const int i = w + kWgWaves * j;
      const bool isy = kWgWaves * j < C::YL;  // (the same for every wave)
      dma16(isy ? ry : rx, voff[j] + (uint32_t)s * (isy ? ystep : xstep), lds0 + (uint32_t)(slot * C::STAGE + i * 1024));
    }
  };

  // transpose reads: lane (g, l16) addresses 4 columns of row 4 g + l16 / 4 (+ 8, + 16 h); 32-column block b of a row
  // sits at 64 (b ^ (row mod 4)) within its 256 bytes
  const int g = lane >> 5, l16 = lane & 15, r2 = l16 >> 2;
  const int in64 = 32 * ((lane >> 4) & 1) + 8 * (l16 & 3);
  const int row0 = 4 * g + r2;
  int ay[C::NB], ax[C::KB];
#pragma unroll
  for (int i = 0; i < C::NB; ++i) {
    const int b = wn * C::NB + i;
    ay[i] = row0 * C::YB + 256 * (b >> 2) + 64 * ((b & 3) ^ r2) + in64;
  }
#pragma unroll
  for (int j = 0; j < C::KB; ++j) {
    const int b = wk * C::KB + j;
    ax[j] = C::XOFF + row0 * C::XB + 256 * (b >> 2) + 64 * ((b & 3) ^ r2) + in64;
  }
  struct Frags {
    bf16x8 y[C::NB], x[C::KB];
  };
  auto tr = [&](const unsigned char* a, int hi) -> bf16x8 {
    const s16x4w lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4w*)a);
    const s16x4w hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4w*)(a + hi));
    const u32x2 l = __builtin_bit_cast(u32x2, lo4), h = __builtin_bit_cast(u32x2, hi4);
    return as_bf16x8(u32x4{l[0], l[1], h[0], h[1]});
  };
  auto read = [&](int slot, int h, Frags& f) {
    const unsigned char* st = wg_lds + slot * C::STAGE;
#pragma unroll
    for (int j = 0; j < C::KB; ++j) f.x[j] = tr(st + ax[j] + 16 * h * C::XB, 8 * C::XB);
#pragma unroll
    for (int i = 0; i < C::NB; ++i) f.y[i] = tr(st + ay[i] + 16 * h * C::YB, 8 * C::YB);
  };
  f32x16 acc[C::NB][C::KB];
#pragma unroll
  for (int i = 0; i < C::NB; ++i)
#pragma unroll
    for (int j = 0; j < C::KB; ++j) acc[i][j] = f32x16{};
  auto multiply = [&](const Frags& f) {
#pragma unroll
    for (int i = 0; i < C::NB; ++i)
#pragma unroll
      for (int j = 0; j < C::KB; ++j) acc[i][j] = mfma32(f.y[i], f.x[j], acc[i][j]);
  };
  // a last stage that is not full: its rows past the segment's end become zero in both tiles (loads past the
  // descriptors leave what the slot held before)
  const int tail = rows - (n_st - 1) * kWgSt;
  auto zero_tail = [&](int slot) {
    unsigned char* st = wg_lds + slot * C::STAGE;
    const u32x4 z{0u, 0u, 0u, 0u};
    for (int c = tid; c < (kWgSt - tail) * (C::YB / 16); c += 64 * kWgWaves) sts16(st + tail * C::YB + 16 * c, z);
    for (int c = tid; c < (kWgSt - tail) * (C::XB / 16); c += 64 * kWgWaves)
      sts16(st + C::XOFF + tail * C::XB + 16 * c, z);
    __syncthreads();
  };

#pragma unroll
  for (int s = 0; s < kWgRing; ++s)
    if (s < n_st) issue(s, s);
  // stage 0 has landed when only the later stages' loads are in flight
  if (n_st >= kWgRing) wg_wait_vmem<(kWgRing - 1) * C::LOADS>();
  else wg_wait_vmem<0>();
  __syncthreads();
  if (n_st == 1 && tail < kWgSt) zero_tail(0);
  Frags f0, f1;
  read(0, 0, f0);
  int slot = 0, s = 0;
  // A stage: its second half is read under the first half's products; at the barrier every wave holds the whole stage
  // in registers, so its slot takes stage s + 4, and stage s + 1, landed (only s + 2 and s + 3 in flight), is read
  // under the second half's products.  The steady loop has no branch: joined with a path that skips the reads, the
  // compiler made the second half's products wait for the next stage's reads.
  for (; s + kWgRing < n_st; ++s) {
    read(slot, 1, f1);
    multiply(f0);
    wg_wait_vmem<2 * C::LOADS>();
    __syncthreads();
    issue(s + kWgRing, slot);
    slot = slot + 1 == kWgRing ? 0 : slot + 1;
    read(slot, 0, f0);
    multiply(f1);
  }
  for (; s + 1 < n_st; ++s) {  // the last stages: nothing left to issue
    read(slot, 1, f1);
    multiply(f0);
    wg_wait_vmem<0>();
    __syncthreads();
    slot = slot + 1 == kWgRing ? 0 : slot + 1;
    if (s + 2 == n_st && tail < kWgSt) zero_tail(slot);
    read(slot, 0, f0);
    multiply(f1);
  }
  read(slot, 1, f1);
  multiply(f0);
  multiply(f1);

  // lane l holds column k = l % 32 and rows n = 8 q + 4 (l / 32) + [0, 4) of a block in quad q
  const int l32 = lane & 31;
  if (p.S > 1) {
    f32x4* const dst = reinterpret_cast<f32x4*>(p.part) + ((int64_t)(sg * tiles + tile) * (C::TN * C::TK / 4)) +
                       w * (C::NB * C::KB * 256) + lane;
#pragma unroll
    for (int i = 0; i < C::NB; ++i)
#pragma unroll
      for (int j = 0; j < C::KB; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          dst[((i * C::KB + j) * 4 + q) * 64] =
              f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
    return;
  }
#pragma unroll
  for (int i = 0; i < C::NB; ++i)
#pragma unroll
    for (int j = 0; j < C::KB; ++j) {
      const int k = k0 + (wk * C::KB + j) * 32 + l32;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int n = n0 + (wn * C::NB + i) * 32 + 8 * (r >> 2) + 4 * g + (r & 3);
        if (n < p.N && k < p.K) {
          if (p.out_f32) ((float*)p.out)[n * p.ldo + k] = acc[i][j][r];
          else ((bf16*)p.out)[n * p.ldo + k] = (bf16)acc[i][j][r];
        }
      }
    }
}

// dW = the segments' partials added in segment order: a thread owns one quad (4 n of one k), reads its S copies 8 at a
// time (16 bytes a lane, whole KiB a wave) and stores 128 (fp32) contiguous bytes per 32 lanes and row.  HBM / last-level
// cache bound: S x the tiles' bytes read once.
template <class C>
__global__ __launch_bounds__(256) void wgrad_reduce_kernel(WgParams p) {
  constexpr int QT = C::TN * C::TK / 4;  // quads per tile
  const int tiles = p.nt * p.kt;
  const int64_t at = (int64_t)blockIdx.x * 256 + threadIdx.x;  // the grid covers tiles * QT exactly
  const int tile = (int)(at / QT), u = (int)(at % QT);
  const int lane = u & 63, q = (u >> 6) & 3, blk = (u >> 8) % (C::NB * C::KB), w = (u >> 8) / (C::NB * C::KB);
  const int i = blk / C::KB, j = blk % C::KB;
  const int n = (tile % p.nt) * C::TN + (w % C::WN * C::NB + i) * 32 + 8 * q + 4 * (lane >> 5);
  const int k = (tile / p.nt) * C::TK + (w / C::WN * C::KB + j) * 32 + (lane & 31);
  if (n >= p.N || k >= p.K) return;
  const f32x4* src = reinterpret_cast<const f32x4*>(p.part) + at;
  const int64_t step = (int64_t)tiles * QT;
  f32x4 sum{0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < p.S; s0 += 8) {
    f32x4 v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = src[min(s0 + e, p.S - 1) * step];
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (s0 + e < p.S) sum += v[e];
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (n + e < p.N) {
      if (p.out_f32) ((float*)p.out)[(n + e) * p.ldo + k] = sum[e];
      else ((bf16*)p.out)[(n + e) * p.ldo + k] = (bf16)sum[e];
    }
}

typedef WgCfg<256, 256, 2> WgWide;    // wave 128 x 64
typedef WgCfg<256, 128, 4> WgNarrow;  // wave 64 x 64

static int wg_check(const mla_weight_grad_args* a) {
  const char* op = "mla_weight_grad";
  MLA_CHECK(a, MLA_ERR_INVALID_ARG, "%s: null args", op);
  MLA_CHECK(a->M > 0 && a->N > 0 && a->K > 0 && a->M < (1 << 24) && a->N < (1 << 20) && a->K < (1 << 20),
            MLA_ERR_INVALID_ARG, "%s: size out of range", op);
  MLA_CHECK(a->N % 8 == 0 && a->K % 8 == 0, MLA_ERR_UNSUPPORTED, "%s: N = %lld and K = %lld must be multiples of 8", op,
            (long long)a->N, (long long)a->K);
  MLA_CHECK(a->dy && a->x && a->dw, MLA_ERR_INVALID_ARG, "%s: null pointer", op);
  MLA_CHECK(((uintptr_t)a->dy & 15) == 0 && ((uintptr_t)a->x & 15) == 0 && ((uintptr_t)a->dw & 3) == 0,
            MLA_ERR_INVALID_ARG, "%s: dy and x must be 16-byte aligned, dw 4-byte aligned", op);
  MLA_CHECK(a->dy_stride >= a->N && a->x_stride >= a->K && a->dw_stride >= a->K && a->dy_stride % 8 == 0 &&
                a->x_stride % 8 == 0,
            MLA_ERR_INVALID_ARG, "%s: row strides must cover a row and be multiples of 8 (dy, x)", op);
  MLA_CHECK(a->dw_dtype == MLA_DTYPE_F32 || a->dw_dtype == MLA_DTYPE_BF16, MLA_ERR_UNSUPPORTED, "%s: dw dtype", op);
  // (before the product below, which a stride near 2^63 would wrap; element offsets of dw stay far below it too)
  MLA_CHECK(a->dy_stride < (1 << 30) && a->x_stride < (1 << 30) && a->dw_stride < (1ll << 40), MLA_ERR_UNSUPPORTED,
            "%s: row stride too large", op);
  // 32-bit byte offsets within a segment (and the stages the ring addresses past it)
  MLA_CHECK((a->M + 8 * kWgSt) * std::max(a->dy_stride, a->x_stride) * 2 < (1ll << 31), MLA_ERR_UNSUPPORTED,
            "%s: operands of 2 GiB or more", op);
  return MLA_OK;
}

template <class C>
static int wg_launch(const WgParams& p, hipStream_t s) {
  wgrad_kernel<C><<<dim3((unsigned)(p.nt * p.kt * p.S)), dim3(64 * kWgWaves), 0, s>>>(p);
  MLA_TRY(launch_status("mla_weight_grad"));
  if (p.S > 1) {
    wgrad_reduce_kernel<C><<<dim3((unsigned)(p.nt * p.kt * (C::TN * C::TK / 1024))), dim3(256), 0, s>>>(p);
    MLA_TRY(launch_status("mla_weight_grad"));
  }
  return MLA_OK;
}

}  // namespace mla

using namespace mla;

extern "C" size_t mla_weight_grad_workspace_bytes(const mla_weight_grad_args* a) {
  // 0 for the sizes mla_weight_grad rejects
  if (!a || a->M <= 0 || a->N <= 0 || a->K <= 0 || a->M >= (1 << 24) || a->N >= (1 << 20) || a->K >= (1 << 20)) return 0;
  return (size_t)wg_plan(a->M, a->N, a->K).part_bytes;
}

extern "C" int mla_weight_grad(const mla_weight_grad_args* a, void* stream) {
  MLA_TRY(wg_check(a));
  const WgPlan pl = wg_plan(a->M, a->N, a->K);
  MLA_CHECK(pl.part_bytes == 0 || (a->workspace && a->workspace_bytes >= (size_t)pl.part_bytes &&
                                   ((uintptr_t)a->workspace & 15) == 0),
            MLA_ERR_WORKSPACE, "mla_weight_grad: workspace of %lld bytes (16-byte aligned) needed, %zu given",
            (long long)pl.part_bytes, a->workspace_bytes);
  WgParams p{(const bf16*)a->dy, (const bf16*)a->x, a->dw, (float*)a->workspace, (int)a->M, (int)a->N, (int)a->K,
             a->dy_stride, a->x_stride, a->dw_stride, pl.S, pl.seg, pl.nt, pl.kt, a->dw_dtype == MLA_DTYPE_F32 ? 1 : 0};
  return pl.narrow ? wg_launch<WgNarrow>(p, (hipStream_t)stream) : wg_launch<WgWide>(p, (hipStream_t)stream);
}
