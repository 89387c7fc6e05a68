// RMSNorm fused into the down-projection GEMM (gfx950): the block's norm1 in front of
// q_down / qk_rope / kv_down (transformer.py:16-27 at :338, then :208-213):
//   r[m]    = 1 / sqrt(sum_k x[m][k]^2 / K + eps)
//   xn[m][k] = bf16((x[m][k] r[m]) w[k])                       (fp32 arithmetic)
//   y[m][n] = bf16( sum_k xn[m][k] W[n][k] )                    (fp32 accumulation)
// the reference's fused kernel (fused_mla_triton_kernels.py:105-230) and its numerics: a first
// pass over x forms r (norm_rms_kernel, 4 bytes per row out), the GEMM streams x again and
// normalises each tile in LDS before its products.  The normalised rows never reach memory.
//
// GEMM.  The product runs transposed, C^T [N][M] = W . xn^T, on v_mfma_f32_32x32x16_bf16: a lane's accumulators hold 4
// consecutive n of one row m (8-byte stores).  A workgroup computes BN (n) x BM (m) outputs with 8 waves, two per SIMD.
// K advances in stages of 32; both operand tiles of a stage (rows of 64 bytes) arrive by direct-to-LDS loads into a
// 4-stage ring, and stage s + 1 is normalised in place while stage s is multiplied.  A row's 4 chunks sit at position
// c ^ ((row / 4) mod 4), so 16 rows x one chunk, which both the fragment reads and the normalisation read, are free of
// bank conflicts.  The finished tile goes through LDS as bf16 rows [m][n], so stores are whole row segments.
//
// What bounds it: a 256 x 256 stage is 1024 MFMA clocks a SIMD, and its LDS traffic (96 KiB of fragments, the
// normalisation's round trip, 32 KiB arriving) comes close to that, with the normalisation's 112 VALU instructions a SIMD
// beside both.  So:
//   * a wave normalises one chunk column (k offset) of the tile, whose 8 norm weights are then the wave's own: they come
//     by scalar loads.  Chunks in tile order took four 16-byte LDS reads of weights per thread and stage, as many bytes
//     as the x fragments;
//   * the one barrier of a stage lies between its two 16-wide halves: the first half's products run under the second
//     half's reads and the normalisation, the next stage's first reads under the second half's products, and the steady
//     loop has no branch.  With one barrier at the end of a stage every read waited behind it;
//   * the tile is chosen for the rounds of 256 workgroups (nl_plan in plans.h): M = 24576, N = 2624 made 1056 tiles of
//     256 x 256, a fifth round of 32 workgroups, where the last 64 columns are now tiles of their own, a quarter as long.
// Measured (kernel trace of 40 calls, medians, the row pass included; one run each on one box), before -> now: 24576 x 2624 x
// 2048 391 -> 341 us (327 with warm clocks), 12288 x 2560 x 1792 147 -> 134, 6555 x 2496 x 1440 113 -> 92, 2735 x 2000 x 1632
// 66 -> 41, 1000 x 2624 x 2048 71 -> 40, 700 x 512 x 1056 38 -> 18.  MfmaUtil at the first 33.4 -> 41.0 %.
#include <cmath>

#include "mla_common.h"

namespace mla {

struct NlParams {
  const bf16* x;         // [M][K], row stride xs
  const bf16* w;         // W [N][K], row stride ws (nn.Linear weights, concatenated)
  const float* wn;       // norm weight [K]
  bf16* y;               // [M][N], row stride ys
  float* inv_rms;        // [M]: written by norm_rms_kernel, read by norm_linear_kernel
  int M, N, K, xs, ws, ys;
  float inv_k, eps;
};

constexpr int kNlStages = 4;   // LDS ring depth
constexpr int kNlWaves = 8;
constexpr int kNlMaxK = 4096;

// BN x BM outputs per workgroup, WN waves along n and 8 / WN along m
template <int BN_, int BM_, int WN_>
struct NlCfg {
  static constexpr int BN = BN_, BM = BM_, WN = WN_, WM = kNlWaves / WN_;
  static constexpr int NB = BN / WN / 32, XJ = BM / WM / 32;  // 32 x 32 blocks per wave
  static constexpr int XOFF = BN * kNlBK * 2;                 // the x tile within a stage
  static constexpr int STAGE = (BN + BM) * kNlBK * 2;
  static constexpr int LOADS = STAGE / 1024 / kNlWaves;
  static constexpr int WL = XOFF / 1024;                      // the stage's first WL loads are W's
  static constexpr int NCH = BM / 128;                        // x chunks a thread normalises per stage
  static constexpr int VPM = NB * XJ > 2 ? 32 * NCH / (NB * XJ - 2) : 1;  // VALU instructions between products
  static constexpr int ES = BN * 2 + 16;                      // epilogue row stride (bytes)
  static constexpr int LDS = kNlStages * STAGE > BM * ES ? kNlStages * STAGE : BM * ES;
  static_assert(STAGE % (1024 * kNlWaves) == 0 && WL % kNlWaves == 0 && BM % 128 == 0 && LDS <= 160 * 1024, "tile shape");
};

__device__ __forceinline__ int nl_swz(int row) { return (row >> 2) & 3; }

template <int N>
__device__ __forceinline__ void nl_wait_vmem() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// r[m] of 4 rows per workgroup, one wave per row: lane l sums the squares of 16-byte chunks
// l, l + 64, ... of the row in fp32, then a butterfly over the wave
__global__ __launch_bounds__(256) void norm_rms_kernel(NlParams p) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= p.M) return;  // wave-uniform; no barrier follows
  const bf16* xr = p.x + (int64_t)row * p.xs;
  float ss = 0.f;
  for (int c = lane; c < p.K / 8; c += 64) {
    const u32x4 v = ldg16(xr + 8 * c);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float lo = lo_bf16(v[e]), hi = hi_bf16(v[e]);
      ss += lo * lo;
      ss += hi * hi;
    }
  }
#pragma unroll
  for (int s = 32; s >= 1; s >>= 1) ss += wave_shfl_xor(ss, s);
  if (lane == 0) p.inv_rms[row] = 1.f / sqrtf(ss * p.inv_k + p.eps);
}

template <class C>
__device__ __forceinline__ void norm_linear_tile(const NlParams& p, int n0, int m0, unsigned char* lds) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = w % C::WN, wm = w / C::WN;
  const int l32 = lane & 31, hk = lane >> 5;

  // direct-to-LDS loads: rows 0 .. BN - 1 of a stage are W rows n0 + row, the rest x rows m0 + row - BN; a load covers 16
  // rows, lane q: row q / 4, position q % 4, which holds the row's chunk (q % 4) ^ swz(row).  Rows past N or M read zero
  // (the descriptors end at the last valid row) and their outputs are not stored.
  const int nv = min(C::BN, p.N - n0), mv = min(C::BM, p.M - m0);
  const buf_rsrc rw = make_rsrc(p.w + (int64_t)n0 * p.ws, rows_bytes(nv, p.ws, p.K * 2));
  const buf_rsrc rx = make_rsrc(p.x + (int64_t)m0 * p.xs, rows_bytes(mv, p.xs, p.K * 2));
  const uint32_t lds0 = lds_addr(lds);
  uint32_t voff[C::LOADS];  // byte offsets at k = 0 of this lane's chunk in each of the wave's loads
#pragma unroll
  for (int j = 0; j < C::LOADS; ++j) {
    const bool isw = kNlWaves * j < C::WL;
    const int i = w + kNlWaves * j;
    const int row = 16 * (isw ? i : i - C::WL) + (lane >> 2);
    voff[j] = (uint32_t)(row * (isw ? p.ws : p.xs) * 2 + ((lane & 3) ^ nl_swz(row)) * 16);
  }
  auto issue = [&](int s, int slot) {
#pragma unroll
    for (int j = 0; j < C::LOADS; ++j)
      dma16(kNlWaves * j < C::WL ? rw : rx, voff[j] + (uint32_t)(s * kNlBK * 2),
            lds0 + (uint32_t)(slot * C::STAGE + (w + kNlWaves * j) * 1024));
  };

  // the normalisation: wave w takes chunk column cw of rows 64 (w / 4) + lane (+ 128), with r of its rows in registers and
  // the column's 8 norm weights in scalar registers
  const int cw = w & 3;
  float rn[C::NCH];
  int noff[C::NCH];
#pragma unroll
  for (int i = 0; i < C::NCH; ++i) {
    const int row = 64 * (w >> 2) + lane + 128 * i;
    noff[i] = C::XOFF + row * 64 + (cw ^ nl_swz(row)) * 16;
    rn[i] = m0 + row < p.M ? p.inv_rms[m0 + row] : 0.f;
  }
  typedef const __attribute__((address_space(4))) float* const_floats;  // constant memory: scalar loads
  const const_floats wn_c = (const_floats)(uintptr_t)(p.wn + 8 * cw);
  float wk[8];  // the norm weights of the next stage to be normalised
  auto load_wk = [&](int s) {
#pragma unroll
    for (int e = 0; e < 8; ++e) wk[e] = wn_c[s * kNlBK + e];
  };
  // (a scalar load in flight makes every LDS wait a full one, so it is waited for under the products before any)
  auto land_wk = [&]() {
    asm volatile("" : "+s"(wk[0]), "+s"(wk[1]), "+s"(wk[2]), "+s"(wk[3]), "+s"(wk[4]), "+s"(wk[5]), "+s"(wk[6]),
                      "+s"(wk[7]));
  };
  auto normalise = [&](int slot) {
    unsigned char* st = lds + slot * C::STAGE;
    u32x4 v[C::NCH], o[C::NCH];
#pragma unroll
    for (int i = 0; i < C::NCH; ++i) v[i] = lds16(st + noff[i]);
#pragma unroll
    for (int i = 0; i < C::NCH; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        o[i][e] = pack_bf16x2((lo_bf16(v[i][e]) * rn[i]) * wk[2 * e], (hi_bf16(v[i][e]) * rn[i]) * wk[2 * e + 1]);
#pragma unroll
    for (int i = 0; i < C::NCH; ++i) sts16(st + noff[i], o[i]);
  };

  // fragment reads: W block i (32 rows), x block j (32 rows), k16 half h: lane (l32, hk) reads row l32, chunk 2 h + hk
  int offw[2], offx[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int rw_ = 32 * C::NB * wn + l32;  // the block's row within the tile is + 32 i (swz unchanged)
    offw[h] = rw_ * 64 + (((2 * h + hk) ^ nl_swz(rw_)) * 16);
    const int rx_ = 32 * C::XJ * wm + l32;
    offx[h] = C::XOFF + rx_ * 64 + (((2 * h + hk) ^ nl_swz(rx_)) * 16);
  }
  struct Frags {
    bf16x8 w[C::NB], x[C::XJ];
  };
  auto read = [&](int slot, int h, Frags& f) {
    const unsigned char* st = lds + slot * C::STAGE;
#pragma unroll
    for (int j = 0; j < C::XJ; ++j) f.x[j] = as_bf16x8(lds16(st + offx[h] + j * 32 * 64));
#pragma unroll
    for (int i = 0; i < C::NB; ++i) f.w[i] = as_bf16x8(lds16(st + offw[h] + i * 32 * 64));
  };
  f32x16 acc[C::NB][C::XJ];
#pragma unroll
  for (int i = 0; i < C::NB; ++i)
#pragma unroll
    for (int j = 0; j < C::XJ; ++j) acc[i][j] = f32x16{};
  auto multiply = [&](const Frags& f) {
#pragma unroll
    for (int i = 0; i < C::NB; ++i)
#pragma unroll
      for (int j = 0; j < C::XJ; ++j) acc[i][j] = mfma32(f.w[i], f.x[j], acc[i][j]);
  };

  const int n_st = p.K / kNlBK;
#pragma unroll
  for (int s = 0; s < kNlStages; ++s)
    if (s < n_st) issue(s, s);
  // stages 0 and 1 have landed when at most stages 2 and 3 are in flight
  if (n_st >= kNlStages) nl_wait_vmem<2 * C::LOADS>();
  else nl_wait_vmem<0>();
  load_wk(0);
  __syncthreads();
  normalise(0);
  load_wk(min(1, n_st - 1));
  __syncthreads();

  Frags f0, f1;
  read(0, 0, f0);
  land_wk();
  int slot = 0, s = 0;
  // At the barrier every wave holds stage s in registers, so its slot takes stage s + 4; stage s + 1 is normalised and
  // stage s + 2, normalised next, has landed (only s + 3 in flight).
  for (; s + kNlStages < n_st; ++s) {
    const int next = slot + 1 == kNlStages ? 0 : slot + 1;
    read(slot, 1, f1);
    multiply(f0);
    normalise(next);
    // the reads first, the normalisation's VALU between the products
    __builtin_amdgcn_sched_group_barrier(0x100, C::NB + C::XJ + C::NCH, 0);  // LDS reads
    __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);                       // MFMA
#pragma unroll
    for (int i = 0; i < C::NB * C::XJ - 2; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x002, C::VPM, 0);  // VALU
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    nl_wait_vmem<C::LOADS>();
    __syncthreads();
    load_wk(s + 2);
    issue(s + kNlStages, slot);
    slot = next;
    read(slot, 0, f0);
    multiply(f1);
    __builtin_amdgcn_sched_barrier(0);
    land_wk();
  }
  for (; s + 1 < n_st; ++s) {  // the last stages: nothing left to issue
    const int next = slot + 1 == kNlStages ? 0 : slot + 1;
    read(slot, 1, f1);
    multiply(f0);
    normalise(next);
    nl_wait_vmem<0>();
    __syncthreads();
    load_wk(min(s + 2, n_st - 1));
    slot = next;
    read(slot, 0, f0);
    multiply(f1);
    land_wk();
  }
  read(slot, 1, f1);
  multiply(f0);
  multiply(f1);
  __syncthreads();  // every wave is done with the ring

  // ---- epilogue: the tile as bf16 rows [m][n] in LDS, then whole row segments stored with 8-byte writes
#pragma unroll
  for (int j = 0; j < C::XJ; ++j) {
    unsigned char* er = lds + (32 * (C::XJ * wm + j) + l32) * C::ES;
#pragma unroll
    for (int i = 0; i < C::NB; ++i) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        // accumulator rows 8 g + 4 hk + [0, 4) of block i
        const f32x16& a = acc[i][j];
        sts8(er + (32 * (C::NB * wn + i) + 8 * g + 4 * hk) * 2,
             u32x2{pack_bf16x2(a[4 * g], a[4 * g + 1]), pack_bf16x2(a[4 * g + 2], a[4 * g + 3])});
      }
    }
  }
  __syncthreads();
  for (int c = tid; c < C::BM * (C::BN / 4); c += 64 * kNlWaves) {
    const int row = c / (C::BN / 4), n = 4 * (c % (C::BN / 4));
    if (row < mv && n < nv) stg8(p.y + (int64_t)(m0 + row) * p.ys + n0 + n, lds8(lds + row * C::ES + n * 2));
  }
}

// Workgroups [0, n_wide) are tiles of C, n tiles of one m tile consecutive (the x rows they share meet in one XCD's L2:
// hardware places id on XCD id % 8); the rest, launched last, are the n remainder's tiles of R, one per m tile.
template <class C, class R>
__global__ __launch_bounds__(64 * kNlWaves, 1) void norm_linear_kernel(NlParams p, int n_nt, int n_wide) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds[C::LDS > R::LDS ? C::LDS : R::LDS];
  int id = blockIdx.x;
  if (id < n_wide) {
    if ((n_wide & 7) == 0) id = (id & 7) * (n_wide >> 3) + (id >> 3);
    norm_linear_tile<C>(p, (id % n_nt) * C::BN, (id / n_nt) * C::BM, lds);
  } else {
    norm_linear_tile<R>(p, n_nt * C::BN, (id - n_wide) * R::BM, lds);
  }
}

typedef NlCfg<256, 256, 2> NlWide;   // wave 128 n x 64 m
typedef NlCfg<128, 256, 2> NlRest;   // wave 64 x 64: an n remainder of up to 128 beside NlWide tiles
typedef NlCfg<256, 128, 4> NlHalf;   // wave 64 x 64
typedef NlCfg<128, 128, 4> NlSmall;  // wave 32 n x 64 m

}  // namespace mla

using namespace mla;

extern "C" int mla_norm_linear(const mla_norm_linear_args* a, void* stream) {
  const char* op = "mla_norm_linear";
  MLA_CHECK(a, MLA_ERR_INVALID_ARG, "%s: null args", op);
  MLA_CHECK(a->M >= 0 && a->N >= 0 && a->K >= 0, MLA_ERR_INVALID_ARG, "%s: negative size", op);
  MLA_CHECK(a->M < (1ll << 31) && a->N < (1 << 20), MLA_ERR_INVALID_ARG, "%s: size out of range", op);
  if (a->M == 0 || a->N == 0) return MLA_OK;
  MLA_CHECK(a->K > 0 && a->K % kNlBK == 0 && a->K <= kNlMaxK, MLA_ERR_UNSUPPORTED,
            "%s: K = %lld must be a positive multiple of %d up to %d", op, (long long)a->K, kNlBK, kNlMaxK);
  MLA_CHECK(a->N % 4 == 0, MLA_ERR_UNSUPPORTED, "%s: N = %lld must be a multiple of 4", op, (long long)a->N);
  MLA_CHECK(a->x && a->w && a->w_norm && a->y && a->inv_rms, MLA_ERR_INVALID_ARG, "%s: null pointer", op);
  MLA_CHECK(((uintptr_t)a->x & 15) == 0 && ((uintptr_t)a->w & 15) == 0 && ((uintptr_t)a->w_norm & 15) == 0 &&
                ((uintptr_t)a->y & 7) == 0 && ((uintptr_t)a->inv_rms & 3) == 0,
            MLA_ERR_INVALID_ARG, "%s: x, w and w_norm must be 16-byte aligned, y 8-byte aligned", op);
  MLA_CHECK(a->x_stride >= a->K && a->w_stride >= a->K && a->y_stride >= a->N && a->x_stride % 8 == 0 &&
                a->w_stride % 8 == 0 && a->y_stride % 4 == 0,
            MLA_ERR_INVALID_ARG, "%s: row strides must cover a row and be multiples of 8 (x, w) and 4 (y)", op);
  // a tile's 256 rows must be addressable with 32-bit offsets from its first row
  MLA_CHECK(a->x_stride < (1 << 22) && a->w_stride < (1 << 22) && a->y_stride < (1ll << 31), MLA_ERR_INVALID_ARG,
            "%s: row stride too large", op);
  MLA_CHECK(std::isfinite(a->eps) && a->eps >= 0.f, MLA_ERR_INVALID_ARG, "%s: eps must be finite and >= 0", op);
  const NlPlan pl = nl_plan(a->M, a->N, a->K);
  const int64_t n_wg = pl.n_wide + pl.n_rest;
  MLA_CHECK(n_wg < (1ll << 31), MLA_ERR_INVALID_ARG, "%s: grid too large", op);
  NlParams p{(const bf16*)a->x, (const bf16*)a->w, a->w_norm, (bf16*)a->y, a->inv_rms, (int)a->M, (int)a->N, (int)a->K,
             (int)a->x_stride, (int)a->w_stride, (int)a->y_stride, 1.f / (float)a->K, a->eps};
  hipStream_t s = (hipStream_t)stream;
  norm_rms_kernel<<<dim3((unsigned)((a->M + 3) / 4)), dim3(256), 0, s>>>(p);
  MLA_TRY(launch_status(op));
  const dim3 grid((unsigned)n_wg), wg(64 * kNlWaves);
  const int nt = (int)pl.n_nt, nw = (int)pl.n_wide;
  if (pl.kind == 0) norm_linear_kernel<NlWide, NlRest><<<grid, wg, 0, s>>>(p, nt, nw);
  else if (pl.kind == 1) norm_linear_kernel<NlHalf, NlHalf><<<grid, wg, 0, s>>>(p, nt, nw);
  else norm_linear_kernel<NlSmall, NlSmall><<<grid, wg, 0, s>>>(p, nt, nw);
  return launch_status(op);
}
