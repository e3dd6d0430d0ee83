// sdm_train.hip -- the dense parts of a training step around the SDM core: the weight gradient of a map in bfloat16
// (sdm_rt_weight_grad), the backward of the RMS norm (sdm_rt_rms_norm_backward; RMSNorm, experiments/track4/sdmllm/
// track4_sdmllm_models.py:63-71) and the mixer's projection weights packed for its two maps
// (sdm_rt_pack_projection; wk, wq, wg, wv of track4_onesdm_models.py:199-206).
#include "sdm_norm.h"
#include "sdm_reduce.h"

namespace sdmrt {

// ---------------------------------------------------------------------------------------------------------------
// weight_grad_kernel: out[s][n][k] = sum over the tokens t of split s of dy[t][n] x[t][k], bfloat16 in, float32 sums.
// Both operands hold the summed index in their rows, so a product's operands (8 consecutive tokens of one column per
// lane) are columns of the tiles: the tiles are staged in LDS as they lie in memory and read through the LDS
// transpose load (ds_read_b64_tr_b16: the 16 lanes of a group address four tokens x 16 columns, 8 bytes a lane, and
// each receives one column's four tokens).
// Block (split, tile of out), WN x WK waves: a wave holds 32 MI x 64 of the tile in v_mfma_f32_32x32x16_bf16
// accumulators.  Steps of 64 tokens in two LDS buffers: while the products of one step run, the next step's rows (in
// registers since the step before) go to the other buffer and the loads of the one after are issued.  LDS rows are
// padded by 64 bytes, so the eight 32-byte pieces that a half-wave reads (four tokens, two groups of columns) fall on
// different banks.  The blocks of one split are dispatched to the same XCDs (split is the fastest grid index), where
// they walk the same tokens together and share them in L2.
// Tiles of 256 x 256 by eight waves where out has them, since the loads bound it (64 KB per 256 x 256 x 64 step against
// 2,048 cycles of products); 128 x 128 by four waves for narrow maps, where larger ones are mostly padding.
// Few columns of out and many tokens (n = 768 or 2,560, 16,384 tokens) leave the GEMM library with small tiles and no
// split of the sum: 139 us for [2,560 x 768] over 16,384 tokens and 94 us for [768 x 768], here 92 and 46 us with the
// partial sums (0.70 and 0.42 PFLOP/s; the sums' record traffic is 22 us of the two).
constexpr int kWgStep = 64;      // tokens per step
constexpr int kWgMinSteps = 4;   // steps per split at least

typedef short short4v __attribute__((ext_vector_type(4)));

// the operand of one 16-token product step: 8 tokens (8 (lane / 32) + 0 .. 7) of column lane % 32 of 32 columns.
// p: the lane's address for its group's first four tokens
template <int PITCH>
__device__ __forceinline__ bf16x8 tr_operand(const uint16_t* p) {
  typedef __attribute__((address_space(3))) short4v* lds4;
  const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(p));
  const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(p + 4 * PITCH));
  const uint2 a = __builtin_bit_cast(uint2, lo), b = __builtin_bit_cast(uint2, hi);
  return __builtin_bit_cast(bf16x8, make_uint4(a.x, a.y, b.x, b.y));
}

template <int MI, int WN, int WK>
struct WgTile {
  static constexpr int threads = 64 * WN * WK;
  static constexpr int bn = 32 * MI * WN, bk = 64 * WK;       // tile of out
  static constexpr int pa = bn + 32, pb = bk + 32;            // LDS row pitches, elements
  static constexpr int buffer = kWgStep * (pa + pb);          // elements of one step
  static constexpr size_t lds = 2 * sizeof(uint16_t) * buffer;
  static constexpr int la = kWgStep * bn / 8 / threads, lb = kWgStep * bk / 8 / threads;   // 16-byte loads per thread
};

template <int MI, int WN, int WK>
__global__ void __launch_bounds__(64 * WN * WK, 2) weight_grad_kernel(const bf16_t* __restrict__ dy, int64_t dys,
                                                                      const bf16_t* __restrict__ x, int64_t xs,
                                                                      int64_t rows, int n, int k, int64_t split_rows,
                                                                      int tiles_k, float* __restrict__ out) {
  using Tl = WgTile<MI, WN, WK>;
  extern __shared__ __attribute__((aligned(16))) uint16_t wlds[];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int n0 = blockIdx.y / tiles_k * Tl::bn, k0 = blockIdx.y % tiles_k * Tl::bk;
  const int64_t t_begin = blockIdx.x * split_rows;
  const int64_t t_end = min(rows, t_begin + split_rows);
  // staging: thread t moves 16-byte pieces t, t + threads, ... of each operand's step, row by row
  constexpr int ca = Tl::bn / 8, cb = Tl::bk / 8;   // pieces per row; they divide the block
  const int pca = 8 * (tid % ca), pcb = 8 * (tid % cb), tra = tid / ca, trb = tid / cb;
  const bool in_n = n0 + pca < n, in_k = k0 + pcb < k;
  const bf16_t* dyc = dy + (in_n ? n0 + pca : 0);
  const bf16_t* xc = x + (in_k ? k0 + pcb : 0);
  uint4 ra[Tl::la], rb[Tl::lb];
  // loads unconditional at clamped rows and columns, what lies outside masked to zero when staged
  auto fetch = [&](int64_t t0) {
#pragma unroll
    for (int i = 0; i < Tl::la; ++i)
      ra[i] = *reinterpret_cast<const uint4*>(dyc + min(t0 + tra + i * (Tl::threads / ca), t_end - 1) * dys);
#pragma unroll
    for (int i = 0; i < Tl::lb; ++i)
      rb[i] = *reinterpret_cast<const uint4*>(xc + min(t0 + trb + i * (Tl::threads / cb), t_end - 1) * xs);
  };
  auto masked = [](uint4 v, bool keep) {
    const uint32_t m = keep ? 0xffffffffu : 0u;
    return make_uint4(v.x & m, v.y & m, v.z & m, v.w & m);
  };
  auto stage = [&](int buf, int64_t t0) {
    uint16_t* sa = wlds + buf * Tl::buffer;
    uint16_t* sb = sa + kWgStep * Tl::pa;
#pragma unroll
    for (int i = 0; i < Tl::la; ++i)
      *reinterpret_cast<uint4*>(&sa[(tra + i * (Tl::threads / ca)) * Tl::pa + pca]) =
          masked(ra[i], in_n && t0 + tra + i * (Tl::threads / ca) < t_end);
#pragma unroll
    for (int i = 0; i < Tl::lb; ++i)
      *reinterpret_cast<uint4*>(&sb[(trb + i * (Tl::threads / cb)) * Tl::pb + pcb]) =
          masked(rb[i], in_k && t0 + trb + i * (Tl::threads / cb) < t_end);
  };
  // the lane's place in a transpose read: token 8 (lane / 32) + (lane % 16) / 4, columns 16 (lane / 16 % 2) + 4 (lane % 4)
  const int trow = 8 * (lane >> 5) + ((lane & 15) >> 2), tcol = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  const int oa = trow * Tl::pa + tcol + 32 * MI * (w % WN);
  const int ob = kWgStep * Tl::pa + trow * Tl::pb + tcol + 64 * (w / WN);
  floatx16 acc[MI][2];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  if (t_begin < t_end) {
    fetch(t_begin);
    stage(0, t_begin);
    fetch(t_begin + kWgStep);
  }
  lds_barrier();
  int buf = 0;
  for (int64_t t0 = t_begin; t0 < t_end; t0 += kWgStep, buf ^= 1) {
    const uint16_t* base = wlds + buf * Tl::buffer;
#pragma unroll
    for (int s = 0; s < kWgStep / 16; ++s) {
      bf16x8 av[MI], bv[2];
#pragma unroll
      for (int i = 0; i < MI; ++i) av[i] = tr_operand<Tl::pa>(base + oa + 16 * s * Tl::pa + 32 * i);
#pragma unroll
      for (int j = 0; j < 2; ++j) bv[j] = tr_operand<Tl::pb>(base + ob + 16 * s * Tl::pb + 32 * j);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[i], bv[j], acc[i][j], 0, 0, 0);
    }
    if (t0 + kWgStep < t_end) {
      stage(buf ^ 1, t0 + kWgStep);
      fetch(t0 + 2 * kWgStep);
    }
    lds_barrier();
  }
  float* dst = out + static_cast<int64_t>(blockIdx.x) * n * k;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int kc = k0 + 64 * (w / WN) + 32 * j + (lane & 31);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int nr = n0 + 32 * (MI * (w % WN) + i) + 8 * (r / 4) + 4 * (lane >> 5) + r % 4;
        if (nr < n && kc < k) dst[static_cast<int64_t>(nr) * k + kc] = acc[i][j][r];
      }
    }
}

// out[i] = part[0][i] + part[1][i] + ... in split order, four values a thread (n k is a multiple of 64)
__global__ void __launch_bounds__(256) split_sum_kernel(const float4* __restrict__ part, int splits, int64_t items4,
                                                        float4* __restrict__ out) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= items4) return;
  float4 s = part[i];
  for (int q = 1; q < splits; ++q) {
    const float4 v = part[q * items4 + i];
    s.x += v.x;
    s.y += v.y;
    s.z += v.z;
    s.w += v.w;
  }
  out[i] = s;
}

using WgWide = WgTile<4, 2, 4>;     // 256 x 256, one block per compute unit
using WgNarrow = WgTile<2, 2, 2>;   // 128 x 128, two

struct WgradPlan {
  bool wide;
  int tiles_n, tiles_k, splits;
  int64_t split_rows;
};

// Splits of the token sum: enough blocks to fill the chip once, as long as a split keeps kWgMinSteps steps (a shorter
// one spends its time on the partial sums, 4 n k bytes written and read back per split)
WgradPlan wgrad_plan(int64_t rows, int n, int k) {
  WgradPlan g;
  const int64_t steps = (rows + kWgStep - 1) / kWgStep;
  const int64_t most = std::max<int64_t>(1, steps / kWgMinSteps);
  // wide tiles where they leave a block for most of the 256 compute units (n = k = 768: 16,384 rows 46 us wide; 4,096
  // rows, 144 wide blocks, 28 us wide)
  g.wide = n >= WgWide::bn && k >= WgWide::bk &&
           (n + WgWide::bn - 1) / WgWide::bn * static_cast<int64_t>((k + WgWide::bk - 1) / WgWide::bk) * most >= 192;
  const int bn = g.wide ? WgWide::bn : WgNarrow::bn, bk = g.wide ? WgWide::bk : WgNarrow::bk;
  g.tiles_n = (n + bn - 1) / bn;
  g.tiles_k = (k + bk - 1) / bk;
  const int64_t tiles = static_cast<int64_t>(g.tiles_n) * g.tiles_k;
  const int64_t want = std::min(most, std::max<int64_t>(1, (g.wide ? 256 : 512) / tiles));
  const int64_t per = std::max<int64_t>(1, (steps + want - 1) / want);
  g.split_rows = per * kWgStep;
  g.splits = static_cast<int>(std::max<int64_t>(1, (steps + per - 1) / per));
  return g;
}

template <int MI, int WN, int WK>
int launch_wgrad(const WgradPlan& g, const void* dy, int64_t dys, const void* x, int64_t xs, int64_t rows, int n, int k,
                 float* part, hipStream_t st) {
  using Tl = WgTile<MI, WN, WK>;
  static const bool ok = allow_lds(reinterpret_cast<const void*>(&weight_grad_kernel<MI, WN, WK>));
  if (!ok) return lds_err("weight grad");
  hipLaunchKernelGGL((weight_grad_kernel<MI, WN, WK>), dim3(g.splits, g.tiles_n * g.tiles_k), dim3(Tl::threads),
                     Tl::lds, st, static_cast<const bf16_t*>(dy), dys, static_cast<const bf16_t*>(x), xs, rows, n, k,
                     g.split_rows, g.tiles_k, part);
  return check_launch("weight grad");
}

// ---------------------------------------------------------------------------------------------------------------
// rms_norm_backward_kernel: y = x rs w, rs = rsqrt(mean(x^2) + eps), the forward's roundings taken as identities (as
// autograd takes .to()):  dx = rs (g - x rs^2 <g, x> / d) with g = dy w,  dw = sum over rows of dy x rs.
// Half a wave per row as in norm_rows (32 lanes, KC pieces of 8 values);
// each half-wave keeps its rows' dw in registers, the block adds its eight in order and leaves one record.
// Bound: HBM, x and dy in and dx out: 26 us for 16,384 rows of 768, float32 x, bfloat16 dy (125 MB, 26 us at a copy's
// rate).  Op by op in torch (powers, means, products, casts and a column sum, each its own pass) it took about 230 us.
constexpr int kNormBwdBlocks = 512;

template <typename InT, typename DyT, int KC>
__global__ void __launch_bounds__(256) rms_norm_backward_kernel(const InT* __restrict__ x, int64_t xs,
                                                                const DyT* __restrict__ dy, int64_t dys,
                                                                const float* __restrict__ w, int64_t rows, int d,
                                                                float eps, InT* __restrict__ dx, int64_t dxs,
                                                                float* __restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) float red[];   // [8][d]
  const int lane = threadIdx.x & 63, hl = lane & 31;
  const int g = threadIdx.x >> 5;   // the block's half-wave
  float wv[KC][8], acc[KC][8];
#pragma unroll
  for (int q = 0; q < KC; ++q) {
    const int c = 8 * (hl + 32 * q);
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[q][e] = wv[q][e] = 0.f;
    if (c < d) load8<float>(w + c, wv[q]);
  }
  // both halves of a wave take part in the sums: the bound is the wave's first row
  for (int64_t r0 = static_cast<int64_t>(blockIdx.x) * 8 + (g & ~1); r0 < rows; r0 += static_cast<int64_t>(gridDim.x) * 8) {
    const int64_t row = r0 + (g & 1);
    const bool live = row < rows;
    const InT* xr = x + (live ? row : 0) * xs;
    const DyT* yr = dy + (live ? row : 0) * dys;
    Piece8<InT> xp[KC];
    Piece8<DyT> yp[KC];
#pragma unroll
    for (int q = 0; q < KC; ++q) {
      const int c = 8 * (hl + 32 * q);
      if (c < d) {
        xp[q] = load_piece8<InT>(xr + c);
        yp[q] = load_piece8<DyT>(yr + c);
      }
    }
    float xv[KC][8], gv[KC][8];
    float ss = 0.f, dot = 0.f;
#pragma unroll
    for (int q = 0; q < KC; ++q) {
      const int c = 8 * (hl + 32 * q);
      if (c < d) {
        unpack8<InT>(xp[q], xv[q]);
        unpack8<DyT>(yp[q], gv[q]);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          ss = fmaf(xv[q][e], xv[q][e], ss);
          dot = fmaf(gv[q][e] * wv[q][e], xv[q][e], dot);
        }
      }
    }
    ss = half_wave_sum(ss, lane);
    dot = half_wave_sum(dot, lane);
    const float rs = rsqrtf(ss / static_cast<float>(d) + eps);
    const float f = rs * rs * (dot / static_cast<float>(d));
    if (live) {
#pragma unroll
      for (int q = 0; q < KC; ++q) {
        const int c = 8 * (hl + 32 * q);
        if (c < d) {
          float o[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            acc[q][e] = fmaf(gv[q][e], xv[q][e] * rs, acc[q][e]);
            o[e] = rs * (gv[q][e] * wv[q][e] - xv[q][e] * f);
          }
          if (dx) store8<InT>(dx + row * dxs + c, o);
        }
      }
    }
  }
  if (!part) return;
#pragma unroll
  for (int q = 0; q < KC; ++q) {
    const int c = 8 * (hl + 32 * q);
    if (c < d) store8<float>(&red[g * d + c], acc[q]);
  }
  __syncthreads();
  for (int c = threadIdx.x; c < d; c += 256) {
    float s = 0.f;
    for (int q = 0; q < 8; ++q) s += red[q * d + c];
    part[static_cast<int64_t>(blockIdx.x) * d + c] = s;
  }
}

int norm_bwd_blocks(int64_t rows) { return static_cast<int>(std::min<int64_t>((rows + 7) / 8, kNormBwdBlocks)); }

template <typename InT, typename DyT>
int launch_norm_bwd(const void* x, int64_t xs, const void* dy, int64_t dys, const float* w, int64_t rows, int d,
                    float eps, void* dx, int64_t dxs, float* part, hipStream_t st) {
  const dim3 grid(norm_bwd_blocks(rows));
  const size_t lds = part ? 8 * sizeof(float) * d : 0;
#define SDM_RT_NB(KC)                                                                                               \
  hipLaunchKernelGGL((rms_norm_backward_kernel<InT, DyT, KC>), grid, dim3(256), lds, st, static_cast<const InT*>(x), \
                     xs, static_cast<const DyT*>(dy), dys, w, rows, d, eps, static_cast<InT*>(dx), dxs, part)
  switch ((d + 255) / 256) {
    case 1: SDM_RT_NB(1); break;
    case 2: SDM_RT_NB(2); break;
    case 3: SDM_RT_NB(3); break;
    case 4: SDM_RT_NB(4); break;
    case 5: case 6: SDM_RT_NB(6); break;
    default: SDM_RT_NB(8); break;
  }
#undef SDM_RT_NB
  return check_launch("rms norm backward");
}

// ---------------------------------------------------------------------------------------------------------------
// pack_projection_kernel: [wk; wq; wg; zero rows up to ra; wv] (rows of d) in the maps' type, and the matching bias
// (bg on wg's rows, zero elsewhere); 8 values a thread
template <typename SrcT, typename DstT>
__global__ void __launch_bounds__(256) pack_projection_kernel(const SrcT* __restrict__ wk, const SrcT* __restrict__ wq,
                                                              const SrcT* __restrict__ wg, const SrcT* __restrict__ wv,
                                                              const SrcT* __restrict__ bg, int za, int H, int ra, int d,
                                                              DstT* __restrict__ out, DstT* __restrict__ bias) {
  const int per = d / 8;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int row = static_cast<int>(i / per);
  if (row >= ra + d) return;
  const int c = 8 * static_cast<int>(i - static_cast<int64_t>(row) * per);
  const bool gate = row >= 2 * za && row < 2 * za + H && wg;
  const SrcT* src = row < za ? wk + static_cast<int64_t>(row) * d
                    : row < 2 * za ? wq + static_cast<int64_t>(row - za) * d
                    : gate ? wg + static_cast<int64_t>(row - 2 * za) * d
                    : row >= ra ? wv + static_cast<int64_t>(row - ra) * d : nullptr;
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (src) load8<SrcT>(src + c, v);
  store8<DstT>(out + static_cast<int64_t>(row) * d + c, v);
  if (c == 0 && bias) bias[row] = from_f32<DstT>(gate && bg ? to_f32(bg[row - 2 * za]) : 0.f);
}

bool rows16(const void* p, int64_t stride, size_t es) {
  return (reinterpret_cast<uintptr_t>(p) & 15u) == 0 && (stride * static_cast<int64_t>(es)) % 16 == 0;
}

}  // namespace sdmrt

using namespace sdmrt;

extern "C" {

size_t sdm_rt_weight_grad_workspace_bytes(int64_t rows, int32_t n, int32_t k) {
  if (rows < 0 || n <= 0 || k <= 0) return 0;
  const WgradPlan g = wgrad_plan(rows, n, k);
  return g.splits > 1 ? sizeof(float) * g.splits * static_cast<size_t>(n) * k : 0;
}

int sdm_rt_weight_grad(const void* dy, int64_t dy_row_stride, const void* x, int64_t x_row_stride, int64_t rows,
                       int32_t n, int32_t k, float* out, void* workspace, size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  if (rows < 0 || n <= 0 || k <= 0) return set_err(SDM_RT_EINVAL, "weight grad: bad sizes");
  if (n % 8 != 0 || k % 8 != 0) return set_err(SDM_RT_EUNSUPPORTED, "weight grad: n and k must be multiples of 8");
  if (!out || (rows > 0 && (!dy || !x))) return set_err(SDM_RT_EINVAL, "weight grad: dy, x and out must not be NULL");
  if (rows > 0 && (dy_row_stride < n || x_row_stride < k))
    return set_err(SDM_RT_EINVAL, "weight grad: row stride below the row");
  if (!rows16(dy, dy_row_stride, 2) || !rows16(x, x_row_stride, 2) || (reinterpret_cast<uintptr_t>(out) & 15u))
    return set_err(SDM_RT_EUNSUPPORTED, "weight grad: rows must be 16-byte aligned");
  const WgradPlan g = wgrad_plan(rows, n, k);
  const int64_t tiles = static_cast<int64_t>(g.tiles_n) * g.tiles_k;
  if (tiles > 65535) return set_err(SDM_RT_EUNSUPPORTED, "weight grad: n x k too large");
  const size_t need = sdm_rt_weight_grad_workspace_bytes(rows, n, k);
  if (need && (!workspace || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 15u)))
    return set_err(SDM_RT_ENOSPACE, "weight grad: workspace %zu bytes < required %zu", workspace_bytes, need);
  hipStream_t st = static_cast<hipStream_t>(stream);
  float* part = need ? static_cast<float*>(workspace) : out;
  int rc = g.wide ? launch_wgrad<4, 2, 4>(g, dy, dy_row_stride, x, x_row_stride, rows, n, k, part, st)
                  : launch_wgrad<2, 2, 2>(g, dy, dy_row_stride, x, x_row_stride, rows, n, k, part, st);
  if (rc) return rc;
  if (need) {
    const int64_t items4 = static_cast<int64_t>(n) * k / 4;
    hipLaunchKernelGGL(split_sum_kernel, dim3(static_cast<unsigned>((items4 + 255) / 256)), dim3(256), 0, st,
                       static_cast<const float4*>(workspace), g.splits, items4, reinterpret_cast<float4*>(out));
    return check_launch("weight grad sum");
  }
  return SDM_RT_OK;
}

size_t sdm_rt_rms_norm_backward_workspace_bytes(int64_t rows, int32_t d) {
  if (rows <= 0 || d <= 0) return 0;
  return sizeof(float) * norm_bwd_blocks(rows) * static_cast<size_t>(d);
}

int sdm_rt_rms_norm_backward(const void* x, int64_t x_row_stride, sdm_rt_dtype x_dtype, const void* dy,
                             int64_t dy_row_stride, sdm_rt_dtype dy_dtype, int64_t rows, int32_t d, const float* w,
                             float eps, void* dx, int64_t dx_row_stride, float* dw, void* workspace,
                             size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  int rc;
  if ((rc = check_dtype(x_dtype, "x_dtype"))) return rc;
  if ((rc = check_dtype(dy_dtype, "dy_dtype"))) return rc;
  if (d <= 0 || d % 8 != 0 || d > 2048)
    return set_err(SDM_RT_EUNSUPPORTED, "rms norm backward: d = %d must be a multiple of 8 up to 2048", d);
  if (rows < 0) return set_err(SDM_RT_EINVAL, "rows must not be negative");
  if (rows == 0) return set_err(SDM_RT_EUNSUPPORTED, "rms norm backward: no rows");
  if (!x || !dy || !w) return set_err(SDM_RT_EINVAL, "x, dy and w must not be NULL");
  if (x_row_stride < d || dy_row_stride < d || (dx && dx_row_stride < d))
    return set_err(SDM_RT_EINVAL, "row stride < d");
  if (!rows16(x, x_row_stride, x_dtype == SDM_RT_BF16 ? 2 : 4) ||
      !rows16(dy, dy_row_stride, dy_dtype == SDM_RT_BF16 ? 2 : 4) ||
      (dx && !rows16(dx, dx_row_stride, x_dtype == SDM_RT_BF16 ? 2 : 4)) || (reinterpret_cast<uintptr_t>(w) & 15u))
    return set_err(SDM_RT_EUNSUPPORTED, "rms norm backward: rows must be 16-byte aligned");
  const size_t need = sdm_rt_rms_norm_backward_workspace_bytes(rows, d);
  if (dw && (!workspace || workspace_bytes < need))
    return set_err(SDM_RT_ENOSPACE, "rms norm backward: workspace %zu bytes < required %zu", workspace_bytes, need);
  hipStream_t st = static_cast<hipStream_t>(stream);
  float* part = dw ? static_cast<float*>(workspace) : nullptr;
  const bool xb = x_dtype == SDM_RT_BF16, yb = dy_dtype == SDM_RT_BF16;
  rc = xb ? (yb ? launch_norm_bwd<bf16_t, bf16_t>(x, x_row_stride, dy, dy_row_stride, w, rows, d, eps, dx, dx_row_stride, part, st)
                : launch_norm_bwd<bf16_t, float>(x, x_row_stride, dy, dy_row_stride, w, rows, d, eps, dx, dx_row_stride, part, st))
          : (yb ? launch_norm_bwd<float, bf16_t>(x, x_row_stride, dy, dy_row_stride, w, rows, d, eps, dx, dx_row_stride, part, st)
                : launch_norm_bwd<float, float>(x, x_row_stride, dy, dy_row_stride, w, rows, d, eps, dx, dx_row_stride, part, st));
  if (rc || !dw) return rc;
  hipLaunchKernelGGL(reduce_records_kernel<float>, dim3((d + 63) / 64), dim3(64 * kRedGroups), 0, st, part,
                     norm_bwd_blocks(rows), static_cast<int64_t>(d), static_cast<int64_t>(d), dw);
  return check_launch("rms norm weight gradient");
}

int sdm_rt_pack_projection(const void* wk, const void* wq, const void* wg, const void* wv, const void* gate_bias,
                           sdm_rt_dtype src_dtype, int32_t addr_rows, int32_t heads, int32_t first_rows, int32_t d,
                           void* out, void* bias_out, sdm_rt_dtype out_dtype, void* stream) {
  g_err[0] = 0;
  int rc;
  if ((rc = check_dtype(src_dtype, "src_dtype"))) return rc;
  if ((rc = check_dtype(out_dtype, "out_dtype"))) return rc;
  if (!wk || !wq || !wv || !out) return set_err(SDM_RT_EINVAL, "wk, wq, wv and out must not be NULL");
  if (addr_rows <= 0 || heads <= 0 || d <= 0 || d % 8 != 0)
    return set_err(SDM_RT_EUNSUPPORTED, "pack projection: d must be a positive multiple of 8");
  if (first_rows < 2 * addr_rows + (wg ? heads : 0)) return set_err(SDM_RT_EINVAL, "pack projection: first_rows too small");
  if (!rows16(wk, 0, 4) || !rows16(wq, 0, 4) || !rows16(wg, 0, 4) || !rows16(wv, 0, 4) || !rows16(out, 0, 4))
    return set_err(SDM_RT_EUNSUPPORTED, "pack projection: the weights must be 16-byte aligned");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid(static_cast<unsigned>((static_cast<int64_t>(first_rows + d) * (d / 8) + 255) / 256));
#define SDM_RT_PK(S, D)                                                                                               \
  hipLaunchKernelGGL((pack_projection_kernel<S, D>), grid, dim3(256), 0, st, static_cast<const S*>(wk),               \
                     static_cast<const S*>(wq), static_cast<const S*>(wg), static_cast<const S*>(wv),                 \
                     static_cast<const S*>(gate_bias), addr_rows, heads, first_rows, d, static_cast<D*>(out),         \
                     static_cast<D*>(bias_out))
  if (src_dtype == SDM_RT_BF16) {
    if (out_dtype == SDM_RT_BF16) SDM_RT_PK(bf16_t, bf16_t); else SDM_RT_PK(bf16_t, float);
  } else {
    if (out_dtype == SDM_RT_BF16) SDM_RT_PK(float, bf16_t); else SDM_RT_PK(float, float);
  }
#undef SDM_RT_PK
  return check_launch("pack projection");
}

}  // extern "C"
