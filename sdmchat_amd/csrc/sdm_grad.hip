// sdm_grad.hip -- the backward of the run-time SDM core (sdm_rt_forward_train, sdm_rt_backward) and of TrainedSdm's
// table layer (sdm_rt_table_backward).
//
// The gradient of RunTimeSdm.forward (track4_onesdm_models.py:195-274, the part between the projections and wo) for
// picks held fixed (topk and the slot ids carry no gradient).  With K[t][s] = lam^(t-1-s) sum_ij wr[t,i] ww[s,j]
// [sir[t,i] = siw[s,j]] (same segment, s < t), num_t = sum_s K[t][s] V_s, den_t = sum_s K[t][s] and, from the
// read-out norm and the mean, dnum_t and dden_t:
//   X[t][s]   = <dnum_t, V_s> + dden_t
//   dwr[t,i]  = sum_{s<t} lam^(t-1-s) sum_j ww[s,j] [match] X[t][s]  = <dnum_t, mem_t[sir_i]> + dden_t cnt_t[sir_i]
//   dww[s,j]  = sum_{t>s} lam^(t-1-s) sum_i wr[t,i] [match] X[t][s]  = <V_s, B_s[siw_j]> + Bc_s[siw_j]
//   dV_s      = sum_j ww[s,j] B_s[siw_j]
// where mem/cnt is the forward memory and B/Bc the adjoint memory written by the reads (slots sir, weights wr,
// values dnum, counts dden) and read by the writes, in reverse time.  What a chunk of 64 tokens reads of its own writes
// is chunk_grad_kernel's, for both directions; the memory carried over chunks is one kernel, grad_scan_kernel: a strict
// causal scan whose reads return, per pick, the dot of the row read with a per-position vector (and, in reverse, the
// weighted sum of the rows).  The forward direction gives dwr, the reverse direction dww and dV.  Then
// addr_grad_tile_kernel (addr_grad_kernel past 64 sub-keys per half) takes the softmax, gate, address normalisation and
// sub-key products back (pk_address :134-148, prepare :199-207) and grad_sums_kernel sums the parameter gradients in a
// fixed order.
//
// lam * dL/dlam (the gradient with respect to log lam) needs no extra pass: sum_{t,s} (t-1-s) K[t][s] X[t][s]
// = sum_t t P_t - sum_s (s+1) Q_s with P_t = sum_i wr[t,i] dwr[t,i] and Q_s = sum_j ww[s,j] dww[s,j].

#include <hipcub/hipcub.hpp>

#include "sdm_reduce.h"
#include "sdm_scan.h"

namespace sdmrt {

constexpr int kGradScanThreads = 512;   // grad scans: 64 positions x 8 lanes


// ---------------------------------------------------------------------------------------------------------------
// read-out backward: out-norm (finish :243-246) and mean read, per (token, head)
//   y = r * rho * w, rho = rsqrt(mean(r^2) + eps2)      dr = rho w dy - rho^3 r <dy w, r> / dh
//   r = num / (den + eps)                               dnum = dr / (den + eps), dden = -<dr, r> / (den + eps)
// Block (row block, head): 32 tokens at a time, 8 lanes per token; the out-norm weight gradient sum_n dy r rho is
// summed per block into part[rb][h][dh] (in a fixed order).
constexpr int kReadGradRows = 256;   // tokens per block

template <typename DyT, int STEPS>
__global__ void __launch_bounds__(256) read_grad_kernel(const DyT* __restrict__ dy, int64_t dy_stride,
                                                        const float* __restrict__ r, const float* __restrict__ den,
                                                        const float* __restrict__ onorm_w, float* __restrict__ dnum,
                                                        float* __restrict__ dden, float* __restrict__ part,
                                                        int64_t N, int H, int dh, int read_mean, float read_eps,
                                                        float out_eps) {
  __shared__ float red[32][65];
  const int h = blockIdx.y;
  const int g = threadIdx.x >> 3;
  const int l8 = threadIdx.x & 7;
  constexpr int kMaxSteps = STEPS;   // steps of 64 columns: dh <= 64 * STEPS
  float acc[kMaxSteps][8];
#pragma unroll
  for (int k = 0; k < kMaxSteps; ++k)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[k][e] = 0.f;
  const int64_t n_begin = static_cast<int64_t>(blockIdx.x) * kReadGradRows;
  const int64_t rstride = static_cast<int64_t>(H) * dh;
  // the head's out-norm weights, the same for every token: loaded once
  float wrow[kMaxSteps][8];
#pragma unroll
  for (int k = 0; k < kMaxSteps; ++k) {
    const int c = 8 * l8 + 64 * k;
    if (onorm_w && c < dh) {
      load_vals<8, float>(onorm_w + h * dh + c, wrow[k]);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) wrow[k][e] = 1.f;
    }
  }
  for (int i = 0; i < kReadGradRows / 32; ++i) {
    const int64_t n = n_begin + 32 * i + g;
    const bool live = n < N;   // every lane runs the cross-lane sums
    const int64_t nn = live ? n : 0;
    const float* rr = r + nn * rstride + static_cast<int64_t>(h) * dh;
    const DyT* dd = dy + nn * dy_stride + static_cast<int64_t>(h) * dh;
    // issued with the rows; den is null for the sum read, which reads a word of the row instead and ignores it
    const float den_n = *(den ? den + nn * H + h : rr);
    float rv[kMaxSteps][8], gv[kMaxSteps][8];
#pragma unroll
    for (int k = 0; k < kMaxSteps; ++k)
#pragma unroll
      for (int e = 0; e < 8; ++e) rv[k][e] = gv[k][e] = 0.f;
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < kMaxSteps; ++k) {
      const int c = 8 * l8 + 64 * k;
      if (c < dh) {
        load_vals<8, float>(rr + c, rv[k]);
        load_vals<8, DyT>(dd + c, gv[k]);
        if (!live) {
#pragma unroll
          for (int e = 0; e < 8; ++e) rv[k][e] = gv[k][e] = 0.f;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(rv[k][e], rv[k][e], ss);
      }
    }
    float rho = 1.f;
    if (onorm_w) {
      ss = sum8(ss);
      rho = 1.f / sqrtf(ss / static_cast<float>(dh) + out_eps);
      float dot = 0.f;
#pragma unroll
      for (int k = 0; k < kMaxSteps; ++k) {
        const int c = 8 * l8 + 64 * k;
        if (c < dh) {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            acc[k][e] = fmaf(gv[k][e] * rv[k][e], rho, acc[k][e]);
            gv[k][e] *= wrow[k][e];
            dot = fmaf(gv[k][e], rv[k][e], dot);
          }
        }
      }
      dot = sum8(dot);
      const float f = rho * rho * rho * dot / static_cast<float>(dh);
#pragma unroll
      for (int k = 0; k < kMaxSteps; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e) gv[k][e] = rho * gv[k][e] - f * rv[k][e];
    }
    float inv = 1.f, dd_sum = 0.f;
    if (read_mean) {
      inv = 1.f / ((live ? den_n : 0.f) + read_eps);
#pragma unroll
      for (int k = 0; k < kMaxSteps; ++k) {
        const int c = 8 * l8 + 64 * k;
        if (c < dh) {
#pragma unroll
          for (int e = 0; e < 8; ++e) dd_sum = fmaf(gv[k][e], rv[k][e], dd_sum);
        }
      }
      dd_sum = sum8(dd_sum);
    }
    if (live) {
      float* dst = dnum + nn * rstride + static_cast<int64_t>(h) * dh;
#pragma unroll
      for (int k = 0; k < kMaxSteps; ++k) {
        const int c = 8 * l8 + 64 * k;
        if (c < dh) {
          float o[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = gv[k][e] * inv;
          store_vals<8, float>(dst + c, o);
        }
      }
      if (l8 == 0) dden[nn * H + h] = read_mean ? -dd_sum * inv : 0.f;
    }
  }
  if (!onorm_w || !part) return;
  // block sum of the out-norm weight gradient: 64 columns at a time through LDS
#pragma unroll
  for (int k = 0; k < kMaxSteps; ++k) {
    if (64 * k >= dh) break;
#pragma unroll
    for (int e = 0; e < 8; ++e) red[g][8 * l8 + e] = acc[k][e];
    __syncthreads();
    if (threadIdx.x < 64 && 64 * k + static_cast<int>(threadIdx.x) < dh) {
      float s = 0.f;
      for (int q = 0; q < 32; ++q) s += red[q][threadIdx.x];
      part[(static_cast<int64_t>(blockIdx.x) * H + h) * dh + 64 * k + threadIdx.x] = s;
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------------------------------------------
// chain plan: the write side of one chunk of a grad scan, built in parallel before the scan (the write records of the
// forward plan, for the picks the forward kept).  Per (chunk, head, batch row), stride chain_stride(KP) bytes:
//   u32 {n_rec, n_ext, reset mask lo, hi}   (the mask of the chunk's positions that empty the memory before they read)
//   wrec[64][KP]   uint2 {slot | q0 << 16 | xo << 22, c0 | more << 31}: the distinct slots the chunk's kept writers
//                  write, record u at [u % 64][u / 64] (group g applies records g, g + 64, ...); q0 the slot's first
//                  kept writer, c0 = lam^(L-1-q0) w; with more, its later writers are ext[xo], ext[xo + 1], ... up to
//                  the one flagged last.  Unused entries are null records {M, 0}.
//   ext[64 * KP]   uint2 {c = lam^(L-1-q) w, q | last << 31}
__host__ __device__ constexpr int chain_stride(int KP) { return (16 + 2 * 64 * KP * 8 + 255) / 256 * 256; }

// Position p of chunk c of a scan in either direction: the chunks are those of 64 tokens from the sequence's start, the
// reverse scan takes them from the last (which may be short) and each from its last token, so both directions agree
// on which pairs of positions share a chunk.
template <bool REV>
struct ChunkSpan {
  int L, base;   // live positions; the chunk's first token
  __device__ __forceinline__ ChunkSpan(int c, int T, int n_chunks) {
    base = (REV ? n_chunks - 1 - c : c) * kChunk;
    L = min(kChunk, T - base);
  }
  __device__ __forceinline__ int token(int p) const { return base + (p < L ? (REV ? L - 1 - p : p) : 0); }
};

struct ChainArgs {
  const int32_t* w_slot;   // [B][H][T][KP] write picks
  const float* w_wt;
  const uint8_t* reset;    // [B*T] or nullptr
  const float* decay;      // [H]
  unsigned char* chains;   // [B][H][n_chunks][chain_stride]
  int B, T, H, M, kk, n_chunks;
};

// one wave per (chunk, head, batch row); lane p = position p of the chunk (in scan order: REV runs backwards)
template <int KP, bool REV>
__global__ void __launch_bounds__(64) chain_plan_kernel(ChainArgs a) {
  __shared__ __attribute__((aligned(16))) int32_t s_sl[kChunk][KP];   // pads -1
  __shared__ __attribute__((aligned(16))) float s_w[kChunk][KP];
  __shared__ float pw[kChunk + 4];
  extern __shared__ unsigned long long wm[];   // [M] writer masks
  const int c = blockIdx.x;
  const int h = blockIdx.y;
  const int b = blockIdx.z;
  const int p = threadIdx.x;
  const int M = a.M;
  const int kk = a.kk;
  const int T = a.T;
  const ChunkSpan<REV> span(c, T, a.n_chunks);
  const int L = span.L;
  const bool valid = p < L;
  const int t = span.token(p);
  const int64_t prow = ((static_cast<int64_t>(b) * a.H + h) * T + t) * KP;
  const float lam = a.decay[h];
  {
    float v = 1.f, sq = lam;   // lam^p by squaring (exact for lam = 0 and lam = 1)
#pragma unroll
    for (int bit = 0; bit < 6; ++bit) {
      v = ((p >> bit) & 1) ? v * sq : v;
      sq *= sq;
    }
    pw[p] = v;
  }
  // loads unconditional inside the row (a missing position reads row 0, no reset flags read a word of the fades),
  // masked after: all of them in flight together
  int slr[KP];
  float wr[KP];
#pragma unroll
  for (int j = 0; j < KP; ++j) {
    slr[j] = a.w_slot[prow + j];
    wr[j] = a.w_wt[prow + j];
  }
  const bool has = valid && a.reset && (REV ? t + 1 < T : true);   // backwards, a reset at t + 1 separates t from it
  const int64_t ri = static_cast<int64_t>(b) * T + (has ? (REV ? t + 1 : t) : 0);
  const uint8_t rv8 = *(a.reset ? a.reset + ri : reinterpret_cast<const uint8_t*>(a.decay));
#pragma unroll
  for (int j = 0; j < KP; ++j) {
    const bool live = valid && j < kk;
    s_sl[p][j] = live ? ((slr[j] >= 0 && slr[j] < M) ? slr[j] : 0) : -1;
    s_w[p][j] = live ? wr[j] : 0.f;
  }
  const bool rf = has && rv8 != 0;
  const unsigned long long rmask = __ballot(rf);
  const int last = rmask ? 63 - __builtin_clzll(rmask) : -1;   // writers before the chunk's last reset do not reach
  const unsigned long long keep = last >= 0 ? ~((1ull << last) - 1ull) : ~0ull;   // the state
  for (int i = p; i < M; i += 64) wm[i] = 0ull;
  __syncthreads();
  if (valid) {
#pragma unroll
    for (int j = 0; j < KP; ++j) {
      if (j >= kk) break;
      atomicOr(&wm[s_sl[p][j]], 1ull << p);
    }
  }
  __syncthreads();
  auto weight_of = [&](int q, int m) {   // the weight with which position q wrote slot m (pads never match)
    float r = 0.f;
#pragma unroll
    for (int j4 = 0; j4 < KP; j4 += 4) {
      const int4 s4 = *reinterpret_cast<const int4*>(&s_sl[q][j4]);
      const float4 w4 = *reinterpret_cast<const float4*>(&s_w[q][j4]);
      r = s4.x == m ? w4.x : r;
      r = s4.y == m ? w4.y : r;
      r = s4.z == m ? w4.z : r;
      r = s4.w == m ? w4.w : r;
    }
    return r;
  };

  // records owned by this position (first kept writer) and their later writers
  int n_own = 0, n_later = 0, n_chained = 0;
  if (valid) {
#pragma unroll
    for (int j = 0; j < KP; ++j) {
      if (j >= kk) break;
      const unsigned long long mm = wm[s_sl[p][j]] & keep;
      if (mm && __builtin_ctzll(mm) == p) {
        const int later = __builtin_popcountll(mm) - 1;
        ++n_own;
        n_later += later;
        n_chained += later > 0;
      }
    }
  }
  const int inc_own = wave_incl_scan(n_own, p);
  const int inc_later = wave_incl_scan(n_later, p);
  const int inc_chained = wave_incl_scan(n_chained, p);
  const int n_rec = __shfl(inc_own, 63);
  const int n_ext = __shfl(inc_later, 63);
  const int n_chained_all = __shfl(inc_chained, 63);
  unsigned char* plan = a.chains + ((static_cast<int64_t>(b) * a.H + h) * a.n_chunks + c) * chain_stride(KP);
  uint2* wrec = reinterpret_cast<uint2*>(plan + 16);
  uint2* ext = wrec + kChunk * KP;
  if (p == 0)
    *reinterpret_cast<uint4*>(plan) =
        make_uint4(n_rec, n_ext, static_cast<uint32_t>(rmask), static_cast<uint32_t>(rmask >> 32));
#pragma unroll
  for (int k = 0; k < KP; ++k)
    if (p + kChunk * k >= n_rec) wrec[p * KP + k] = make_uint2(static_cast<uint32_t>(M), 0u);
  if (!valid) return;
  // slots with later writers take the lowest record indexes (records k = 0, 1, ... of the groups), so the scan's
  // walks of the later writers gather in the first record batches
  int u_m = inc_chained - n_chained, u_s = n_chained_all + (inc_own - inc_chained) - (n_own - n_chained);
  int e = inc_later - n_later;
#pragma unroll
  for (int j = 0; j < KP; ++j) {
    if (j >= kk) break;
    const int m = s_sl[p][j];
    unsigned long long mm = wm[m] & keep;
    if (!mm || __builtin_ctzll(mm) != p) continue;
    mm &= mm - 1ull;
    const uint32_t cw = __float_as_uint(pw[L - 1 - p] * s_w[p][j]) | (mm ? 0x80000000u : 0u);
    const int u = mm ? u_m++ : u_s++;
    wrec[(u & 63) * KP + (u >> 6)] =
        make_uint2(static_cast<uint32_t>(m) | (static_cast<uint32_t>(p) << 16) | (static_cast<uint32_t>(e) << 22), cw);
    while (mm) {
      const int q = __builtin_ctzll(mm);
      mm &= mm - 1ull;
      ext[e] = make_uint2(__float_as_uint(pw[L - 1 - q] * weight_of(q, m)),
                          static_cast<uint32_t>(q) | (mm ? 0u : 0x80000000u));
      ++e;
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// grad_scan_kernel: the per-pick scan over the carried memory (see the top of this file); what a chunk's positions
// read of the chunk's own writes is chunk_grad_kernel's
struct GradScanArgs {
  const int32_t* r_slot;   // [B][H][T][KP] read picks (entries >= kk ignored)
  const float* r_wt;       //   and weights
  const void* wv;          // write value rows (H * dh per row), type WT
  int64_t wv_stride;
  const float* wc;         // [B*T][H] write count factors, or nullptr for 1
  const void* rv;          // read vector rows, type RT
  int64_t rv_stride;
  const float* rc;         // [B*T][H] read count factors, or nullptr for 1
  const float* decay;      // [H]
  float* dot_out;          // [dh / CW][B][H][T][KP] per-pick dots of this column group (count term in group 0)
  const float* sum_in;     // rows of H * dh added to the sums (chunk_grad_kernel's part); with sum_out
  void* sum_out;           // rows of H * dh (weighted sums of the rows read; float32, bfloat16 with sum_bf16), or nullptr
  int64_t sum_stride;
  int sum_bf16;
  const unsigned char* chains;   // [B][H][n_chunks][chain_stride(KP)] chain plans of the writes (chain_plan_kernel)
  int B, T, H, dh, M, kk, n_chunks;
  int vec;                 // the picks, rows and sums are aligned for one load per lane's piece
};

// CPL elements of a row as one load brings them
template <typename T, int CPL>
struct alignas(sizeof(T) * CPL) RawSeg {
  T e[CPL];
};

// chain entries a grad_scan stages in LDS (the rest are read from the chain plan in global memory); typical chunks
// hold 100-400 entries
__host__ __device__ constexpr int grad_ext_stage(int KP) { return KP <= 8 ? 64 * KP * 8 : 3072; }

__host__ __device__ constexpr size_t align16(size_t x) { return (x + 15) / 16 * 16; }

// LDS of one grad_scan workgroup: slab A[M + 1][CW] and counts cnt[M + 1] (row M stays zero: null write records read
// it and write nothing), the chunk's write values s_wv[64][CW], count factors s_wc[64], fade powers pw[68], write
// records s_rec[64][KP] and staged chain entries
struct GradScanLds {
  size_t A, cnt, wv, wc, pw, rec, ext, total;
  __host__ __device__ constexpr GradScanLds(int M, int KP, int CW)
      : A(0),
        cnt(align16(4 * static_cast<size_t>(M + 1) * CW)),
        wv(cnt + align16(4 * static_cast<size_t>(M + 1))),
        wc(wv + 4 * 64 * CW),
        pw(wc + 4 * 64),
        rec(pw + 4 * 68),
        ext(rec + 8 * 64 * KP),
        total(ext + grad_ext_stage(KP)) {}
};

// weight with which chunk position q wrote slot m >= 0 (0 if it did not); pad picks hold slot -1 and never match
template <int KP>
__device__ __forceinline__ float writer_weight(const int32_t* s_ws, const float* s_ww, int q, int m) {
  float r = 0.f;
#pragma unroll
  for (int j4 = 0; j4 < KP; j4 += 4) {
    const int4 s = *reinterpret_cast<const int4*>(&s_ws[q * KP + j4]);
    const float4 w = *reinterpret_cast<const float4*>(&s_ww[q * KP + j4]);
    r = s.x == m ? w.x : r;
    r = s.y == m ? w.y : r;
    r = s.z == m ? w.z : r;
    r = s.w == m ? w.w : r;
  }
  return r;
}

// The 8 lanes of a group hold partial values p[0..8); lane l8 returns the group sum of p[l8] (a butterfly that
// halves the vector at each step; fixed order).  The exchanges are DPP moves: the mirror within 8 lanes pairs the
// two halves of the group, then the quad permutes pair lanes 2 and 1 apart.
__device__ __forceinline__ float group_reduce_scatter8(const float (&p)[8], int l8) {
  float t4[4], t2[2];
  const bool b2 = l8 & 4, b1 = l8 & 2, b0 = l8 & 1;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float mine = b2 ? p[4 + i] : p[i];
    const float other = b2 ? p[i] : p[4 + i];
    t4[i] = mine + dpp_f<0x141>(other);   // row_half_mirror
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float mine = b1 ? t4[2 + i] : t4[i];
    const float other = b1 ? t4[i] : t4[2 + i];
    t2[i] = mine + dpp_f<0x4e>(other);    // quad_perm [2,3,0,1]
  }
  const float mine = b0 ? t2[1] : t2[0];
  const float other = b0 ? t2[0] : t2[1];
  return mine + dpp_f<0xb1>(other);       // quad_perm [1,0,3,2]
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u(uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, 0xf, 0xf, true));
}

// OR over the aligned group of 8 lanes
__device__ __forceinline__ unsigned long long group_or8(unsigned long long v) {
  uint32_t lo = static_cast<uint32_t>(v), hi = static_cast<uint32_t>(v >> 32);
  lo |= dpp_u<0xb1>(lo);
  hi |= dpp_u<0xb1>(hi);
  lo |= dpp_u<0x4e>(lo);
  hi |= dpp_u<0x4e>(hi);
  lo |= dpp_u<0x141>(lo);
  hi |= dpp_u<0x141>(hi);
  return (static_cast<unsigned long long>(hi) << 32) | lo;
}

// What a chunk's positions read of the chunk's own writes, for both directions at once: with X[t][s] = <dnum_t, V_s> +
// dden_t and c[t][s] = lam^(t-1-s) for s < t of one chunk and one segment,
//   dwr[t,i] += sum_s c ww[s,j] [match] X,  dww[s,j] += sum_t c wr[t,i] [match] X,
//   dV_s      = sum_t c (sum_ij wr[t,i] ww[s,j] [match]) dnum_t
// None of it needs the carried memory, so it runs over all chunks in parallel instead of inside the two scans, whose
// chunks form a chain of 32 steps (B=8, T=2048) on 192 of the 256 compute units: there these loops were two fifths of
// each scan.  B=8, T=2048, 12 heads, k=8, bfloat16: the scans 211 + 209 -> 132 + 143 us, this kernel 53 us; k=16
// float32 (B=5, T=301, 4 heads): 114 + 116 -> 53 + 74, this kernel 19 us.
// Block (chunk, head x group of 64 columns, batch row), 512 threads = 64 positions x 8 lanes of 8 columns.  Each slot's
// writers (then its readers) of the chunk are a 64-bit mask in LDS; a position's lanes walk the union of their picks'
// masks together, in position order (a fixed order), only over pairs that match.  A wave's positions are neighbours:
// the last have the most writers before them and the fewest readers after them, so the two loops balance.
struct ChunkGradArgs {
  const int32_t* slot[2];   // write, read picks [B][H][T][KP] (entries >= kk ignored)
  const float* wt[2];
  const void* v;            // value rows (H * dh per row), type VT
  int64_t v_stride;
  const float* dnum;        // [B*T] rows of H * dh
  const float* dden;        // [B*T][H]
  const uint8_t* reset;     // [B*T] or nullptr
  const float* decay;       // [H]
  float* dot_w;             // [column group][B][H][T][KP] partial dww, dwr (dden term in group 0)
  float* dot_r;
  float* dv;                // rows of H * dh: partial dV
  int B, T, H, dh, M, kk, n_xg;
};

struct ChunkGradLds {
  size_t mask, v, dn, sl, wt, pw, dd, total;
  __host__ __device__ constexpr ChunkGradLds(int M, int KP)
      : mask(0),
        v(align16(8 * static_cast<size_t>(M))),
        dn(v + 4 * 64 * 64),
        sl(dn + 4 * 64 * 64),
        wt(sl + 2 * 4 * 64 * KP),
        pw(wt + 2 * 4 * 64 * KP),
        dd(pw + 4 * 64),
        total(dd + 4 * 64) {}
};

template <int KP, typename VT>
__global__ void __launch_bounds__(kGradScanThreads) chunk_grad_kernel(ChunkGradArgs a) {
  constexpr int NO = KP / 8;   // picks per lane: l8, l8 + 8
  extern __shared__ __attribute__((aligned(16))) unsigned char clds[];
  const ChunkGradLds lay(a.M, KP);
  unsigned long long* mask = reinterpret_cast<unsigned long long*>(clds + lay.mask);
  float* sv = reinterpret_cast<float*>(clds + lay.v);
  float* sdn = reinterpret_cast<float*>(clds + lay.dn);
  int32_t* ssl = reinterpret_cast<int32_t*>(clds + lay.sl);   // [2][64][KP], pads -1
  float* swt = reinterpret_cast<float*>(clds + lay.wt);
  float* pw = reinterpret_cast<float*>(clds + lay.pw);
  float* sdd = reinterpret_cast<float*>(clds + lay.dd);
  const int u0 = blockIdx.x * kChunk;
  const int h = blockIdx.y % a.H, xg = blockIdx.y / a.H;
  const int b = blockIdx.z;
  const int tid = threadIdx.x, p = tid >> 3, l8 = tid & 7, lane = tid & 63;
  const int M = a.M, kk = a.kk, T = a.T;
  const int L = min(kChunk, T - u0);
  const bool valid = p < L;
  const int t = u0 + (valid ? p : 0);
  const int64_t n = static_cast<int64_t>(b) * T + t;
  const int64_t prow = ((static_cast<int64_t>(b) * a.H + h) * T + t) * KP;
  const float lam = a.decay[h];
  // the lane's columns of the position's rows: 4 l8 .. + 3 and 32 + 4 l8 .. + 3 of the group's 64
  float dn[8], v[8];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int c = 64 * xg + 32 * q + 4 * l8;
    float x4[4] = {0.f, 0.f, 0.f, 0.f}, y4[4] = {0.f, 0.f, 0.f, 0.f};
    if (valid && c < a.dh) {
      load_vals<4, float>(a.dnum + n * a.H * a.dh + static_cast<int64_t>(h) * a.dh + c, x4);
      load_vals<4, VT>(static_cast<const VT*>(a.v) + n * a.v_stride + static_cast<int64_t>(h) * a.dh + c, y4);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      dn[4 * q + e] = x4[e];
      v[4 * q + e] = y4[e];
    }
    *reinterpret_cast<float4*>(&sdn[p * 64 + 32 * q + 4 * l8]) = make_float4(x4[0], x4[1], x4[2], x4[3]);
    *reinterpret_cast<float4*>(&sv[p * 64 + 32 * q + 4 * l8]) = make_float4(y4[0], y4[1], y4[2], y4[3]);
  }
  const float dd = valid && xg == 0 ? a.dden[n * a.H + h] : 0.f;
  if (l8 == 0) sdd[p] = dd;
  int sl[2][NO];
  float wt[2][NO];
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int o = 0; o < NO; ++o) {
      const int j = l8 + 8 * o;
      const bool live = valid && j < kk;
      const int s = live ? a.slot[k][prow + j] : 0;
      sl[k][o] = live ? (s >= 0 && s < M ? s : 0) : -1;
      wt[k][o] = live ? a.wt[k][prow + j] : 0.f;
      ssl[(k * 64 + p) * KP + j] = sl[k][o];
      swt[(k * 64 + p) * KP + j] = wt[k][o];
    }
  if (tid < 64) {
    float f = 1.f, sq = lam;   // lam^tid by squaring (exact for lam = 0 and lam = 1)
#pragma unroll
    for (int bit = 0; bit < 6; ++bit) {
      f = ((tid >> bit) & 1) ? f * sq : f;
      sq *= sq;
    }
    pw[tid] = f;
  }
  // the chunk's resets, in every wave
  const uint8_t rv8 = *(a.reset ? a.reset + static_cast<int64_t>(b) * T + u0 + min(lane, L - 1)
                                : reinterpret_cast<const uint8_t*>(a.decay));
  const unsigned long long rmask = __ballot(a.reset && lane < L && rv8 != 0);

  float dot[2][NO], sum[8];
#pragma unroll
  for (int o = 0; o < NO; ++o) dot[0][o] = dot[1][o] = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) sum[e] = 0.f;
  const unsigned long long bit = 1ull << p, below = bit - 1ull, above = ~(below | bit);
  // k = 0: position p reads the writers before it; k = 1: position p's writes are read by the readers after it
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if (k == 1) lds_barrier();   // the writers' masks are done with
    for (int i = tid; i < M; i += kGradScanThreads) mask[i] = 0ull;
    lds_barrier();
#pragma unroll
    for (int o = 0; o < NO; ++o)
      if (sl[k][o] >= 0) atomicOr(&mask[sl[k][o]], bit);
    lds_barrier();
    unsigned long long vis;   // the other side's positions of the segment
    if (k == 0) {
      const unsigned long long upto = rmask & (below | bit);
      vis = below & (upto ? ~((1ull << (63 - __builtin_clzll(upto))) - 1ull) : ~0ull);
    } else {
      const unsigned long long after = rmask & above;
      vis = above & (after ? (after & -after) - 1ull : ~0ull);
    }
    unsigned long long mk[NO], any = 0ull;
#pragma unroll
    for (int o = 0; o < NO; ++o) {
      const int s = sl[1 - k][o];
      mk[o] = s >= 0 ? mask[s] & vis : 0ull;
      any |= mk[o];
    }
    unsigned long long U = group_or8(any);
    const float* rows = k == 0 ? sv : sdn;
    while (U) {
      const int q = __builtin_ctzll(U);
      U &= U - 1ull;
      const float4 x0 = *reinterpret_cast<const float4*>(&rows[q * 64 + 4 * l8]);
      const float4 x1 = *reinterpret_cast<const float4*>(&rows[q * 64 + 32 + 4 * l8]);
      const float xr[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
      const float f = pw[k == 0 ? p - 1 - q : q - 1 - p];
      float X = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) X = fmaf(k == 0 ? dn[e] : v[e], xr[e], X);
      X = sum8(X) + (k == 0 ? dd : sdd[q]);
      float cs = 0.f;
#pragma unroll
      for (int o = 0; o < NO; ++o) {
        const float wq = writer_weight<KP>(ssl + k * 64 * KP, swt + k * 64 * KP, q, sl[1 - k][o]);
        const float co = ((mk[o] >> q) & 1ull) ? f * wq : 0.f;
        dot[1 - k][o] = fmaf(co, X, dot[1 - k][o]);
        cs = fmaf(wt[1 - k][o], co, cs);
      }
      if (k == 1) {
        cs = sum8(cs);
#pragma unroll
        for (int e = 0; e < 8; ++e) sum[e] = fmaf(cs, xr[e], sum[e]);
      }
    }
  }
  if (!valid) return;
  const int64_t cg = static_cast<int64_t>(xg) * a.B * a.H * T * KP;
#pragma unroll
  for (int o = 0; o < NO; ++o) {
    const int j = l8 + 8 * o;
    a.dot_w[cg + prow + j] = dot[0][o];
    a.dot_r[cg + prow + j] = dot[1][o];
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int c = 64 * xg + 32 * q + 4 * l8;
    if (c < a.dh) {
      float o4[4] = {sum[4 * q], sum[4 * q + 1], sum[4 * q + 2], sum[4 * q + 3]};
      store_vals<4, float>(a.dv + n * a.H * a.dh + static_cast<int64_t>(h) * a.dh + c, o4);
    }
  }
}

// One workgroup per (column group, head, batch row): 512 threads = 64 positions x 8 lanes of CW/8 columns; the
// slab A (true state mu * A) and the counts stay in LDS.  REV runs the sequence backwards (ChunkSpan); a reset at t
// then separates t - 1 and earlier from what came before it.  Per chunk of 64 positions:
//   read    group = position: the carried rows of its picks (scaled by mu lam^p; none after a reset in the chunk); per
//           pick the dot with the position's read vector (+ the read count factor times the count, in column group 0)
//           and, with sum_out, the pick-weighted sum of the rows
//   sums    group g takes the chain plan's write records g + 64 k: each written slot's old row plus its kept writers'
//           faded values / mu (mu <- mu lam^L; a chunk with a reset empties the slab), one owner per row, lane l8 the
//           count of record l8 + 8 b
//   store   the rows and counts back, the next chunk's write values, records and chain entries into LDS
// with a barrier before and after the stores.  Bound: the chain of chunks on one compute unit per slab and column
// group (192 of 256 at B=8, 12 heads), 8,500 cycles each: 3,900 of VALU, 2,900 of LDS (a quarter of it bank conflicts of
// the random rows), the rest waits; neither fewer vector-memory instructions nor shorter walks of the chains moved it.
template <int CW, int KP, bool REV, typename WT, typename RT>
__global__ void __launch_bounds__(kGradScanThreads) grad_scan_kernel(GradScanArgs a) {
  constexpr int CPL = CW / 8;
  extern __shared__ __attribute__((aligned(16))) unsigned char glds[];
  const int M = a.M;
  const GradScanLds lay(M, KP, CW);
  float* A = reinterpret_cast<float*>(glds + lay.A);
  float* cnt = reinterpret_cast<float*>(glds + lay.cnt);
  float* s_wv = reinterpret_cast<float*>(glds + lay.wv);
  float* s_wc = reinterpret_cast<float*>(glds + lay.wc);
  float* pw = reinterpret_cast<float*>(glds + lay.pw);
  uint2* s_rec = reinterpret_cast<uint2*>(glds + lay.rec);
  unsigned char* s_ext = glds + lay.ext;
  constexpr int XS = grad_ext_stage(KP);
  constexpr int NX = (XS / 16 + kGradScanThreads - 1) / kGradScanThreads;   // staged chain pieces per thread

  const int cg = blockIdx.x;
  const int h = blockIdx.y;
  const int b = blockIdx.z;
  const int tid = threadIdx.x;
  const int g = tid >> 3;
  const int l8 = tid & 7;
  const int col0 = cg * CW;
  const int kk = a.kk;
  const int T = a.T;
  const int64_t bh = static_cast<int64_t>(b) * a.H + h;
  const float lam = a.decay[h];
  float* dot_out = a.dot_out + (static_cast<int64_t>(cg) * a.B * a.H + bh) * T * KP;

  for (int i = tid; i < (M + 1) * CW; i += kGradScanThreads) A[i] = 0.f;
  for (int i = tid; i <= M; i += kGradScanThreads) cnt[i] = 0.f;
  if (tid <= kChunk) {
    float v = 1.f;   // lam^tid by repeated multiplication (exact for lam = 0 and lam = 1)
    for (int e = 0; e < tid; ++e) v *= lam;
    pw[tid] = v;
  }
  float mu = 1.f;
  __syncthreads();

  // one chunk's global inputs, loaded a chunk ahead into registers (raw element types, converted when used)
  struct In {
    RawSeg<WT, CPL> wv;
    float wc;
    RawSeg<int, 4> rs[KP / 4];
    RawSeg<float, 4> rw[KP / 4];
    RawSeg<RT, CPL> rv;
    float rcf;
    RawSeg<float, CPL> sum;
    uint2 own_w[KP / 8];  // write records k = l8 + 8 b of the group (the lane's count updates; staged for the group)
    uint4 xp[NX];         // chain pieces to stage
    uint2 rm;             // the chunk's reset mask
  };
  const unsigned char* chains = a.chains + bh * a.n_chunks * chain_stride(KP);
  auto fetch = [&](int c, In& x) {
    const ChunkSpan<REV> span(c, T, a.n_chunks);
    const bool valid = g < span.L;
    const int t = span.token(g);   // the chunk's first token stands in for a missing position
    const int64_t n = static_cast<int64_t>(b) * T + t;
    const int64_t prow = (bh * T + t) * KP;
    const int64_t vcol = static_cast<int64_t>(h) * a.dh + col0 + CPL * l8;
    // one load per lane's piece where everything is aligned: 9 loads per wave and chunk instead of 25 to 38
    const WT* wvp = static_cast<const WT*>(a.wv) + n * a.wv_stride + vcol;
    const RT* rvp = static_cast<const RT*>(a.rv) + n * a.rv_stride + vcol;
    const float* sip = REV ? a.sum_in + n * a.H * a.dh + vcol : nullptr;
    if (a.vec) {
      x.wv = *reinterpret_cast<const RawSeg<WT, CPL>*>(wvp);
      x.rv = *reinterpret_cast<const RawSeg<RT, CPL>*>(rvp);
      if constexpr (REV) x.sum = *reinterpret_cast<const RawSeg<float, CPL>*>(sip);
#pragma unroll
      for (int i = 0; i < KP / 4; ++i) {
        x.rs[i] = *reinterpret_cast<const RawSeg<int, 4>*>(a.r_slot + prow + 4 * i);
        x.rw[i] = *reinterpret_cast<const RawSeg<float, 4>*>(a.r_wt + prow + 4 * i);
      }
    } else {
      asm volatile("" ::: "memory");   // keeps the compiler from merging the branches' loads into element loads
#pragma unroll
      for (int k = 0; k < CPL; ++k) {
        x.wv.e[k] = wvp[k];
        x.rv.e[k] = rvp[k];
        if constexpr (REV) x.sum.e[k] = sip[k];
      }
#pragma unroll
      for (int i = 0; i < KP; ++i) {
        x.rs[i / 4].e[i % 4] = a.r_slot[prow + i];
        x.rw[i / 4].e[i % 4] = a.r_wt[prow + i];
      }
    }
    x.wc = valid ? (a.wc ? a.wc[n * a.H + h] : 1.f) : 0.f;
    x.rcf = (valid && a.rc) ? a.rc[n * a.H + h] : 1.f;
    const unsigned char* cp = chains + static_cast<int64_t>(c) * chain_stride(KP);
    x.rm = reinterpret_cast<const uint2*>(cp)[1];
    const uint2* wrow = reinterpret_cast<const uint2*>(cp + 16) + g * KP;
#pragma unroll
    for (int k = 0; k < KP / 8; ++k) x.own_w[k] = wrow[l8 + 8 * k];
    // the first chain entries (the whole staged span: loads past n_ext stay inside the plan)
    const uint4* xs = reinterpret_cast<const uint4*>(cp + 16 + 8 * kChunk * KP);
#pragma unroll
    for (int k = 0; k < NX; ++k) {
      const int piece = tid + k * kGradScanThreads;
      x.xp[k] = piece < XS / 16 ? xs[piece] : make_uint4(0u, 0u, 0u, 0u);
    }
  };

  // a chunk's write values, count factors, records and chain entries into LDS
  auto stage = [&](const In& x, bool valid) {
    float vv[CPL];
#pragma unroll
    for (int k = 0; k < CPL; ++k) vv[k] = valid ? to_f32(x.wv.e[k]) : 0.f;
    lds_seg_store<CPL>(&s_wv[g * CW + CPL * l8], *reinterpret_cast<const Seg<CPL>*>(vv));
    if (l8 == 0) s_wc[g] = x.wc;
#pragma unroll
    for (int k = 0; k < KP / 8; ++k) s_rec[g * KP + l8 + 8 * k] = x.own_w[k];
#pragma unroll
    for (int k = 0; k < NX; ++k) {
      const int piece = tid + k * kGradScanThreads;
      if (piece < XS / 16) reinterpret_cast<uint4*>(s_ext)[piece] = x.xp[k];
    }
  };

  In cur;
  fetch(0, cur);
  stage(cur, g < ChunkSpan<REV>(0, T, a.n_chunks).L);
  lds_barrier();
  for (int c = 0; c < a.n_chunks; ++c) {
    const ChunkSpan<REV> span(c, T, a.n_chunks);
    const int L = span.L;
    const bool valid = g < L;
    const int t = span.token(g);
    const int64_t n = static_cast<int64_t>(b) * T + t;
    const unsigned long long rmask = (static_cast<unsigned long long>(cur.rm.y) << 32) | cur.rm.x;
    // the read side of this position, in registers: all picks (every lane), the lane's vector columns
    int rs[KP];
    float rw[KP];
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      rs[i] = static_cast<int>(min(static_cast<uint32_t>(cur.rs[i / 4].e[i % 4]), static_cast<uint32_t>(M)));
      rw[i] = cur.rw[i / 4].e[i % 4];
    }
    if (kk < KP) {   // pads, as stray slots, read row M, which is zero
#pragma unroll
      for (int i = 0; i < KP; ++i)
        if (i >= kk) {
          rs[i] = M;
          rw[i] = 0.f;
        }
    }
    float rv[CPL];
#pragma unroll
    for (int k = 0; k < CPL; ++k) rv[k] = valid ? to_f32(cur.rv.e[k]) : 0.f;
    const float rcf = cur.rcf;
    In nxt;
    const bool more = c + 1 < a.n_chunks;
    if (more) fetch(c + 1, nxt);   // in flight across the barrier below (it orders LDS only)

    // read
    constexpr int NO = KP / 8;   // picks owned per lane: l8, l8 + 8
    float dot[NO];
#pragma unroll
    for (int o = 0; o < NO; ++o) dot[o] = 0.f;
    float sum[CPL];
#pragma unroll
    for (int k = 0; k < CPL; ++k) sum[k] = 0.f;
    if (valid) {
      const int p = g;
      if (!(rmask & (p == 63 ? ~0ull : (2ull << p) - 1ull))) {   // the carried state
        const float fin = mu * pw[p];
        float part[KP];
#pragma unroll
        for (int i = 0; i < KP; ++i) {
          const Seg<CPL> x = lds_seg<CPL>(&A[rs[i] * CW + CPL * l8]);
          float d = 0.f;
#pragma unroll
          for (int k = 0; k < CPL; ++k) {
            d = fmaf(rv[k], x.v[k], d);
            sum[k] = fmaf(rw[i], x.v[k], sum[k]);
          }
          part[i] = d;
        }
#pragma unroll
        for (int o = 0; o < NO; ++o) {
          float p8[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) p8[e] = part[8 * o + e];
          dot[o] = fin * group_reduce_scatter8(p8, l8);
        }
        if (cg == 0) {   // the count term, once per pick
#pragma unroll
          for (int o = 0; o < NO; ++o) {
            int so = 0;
#pragma unroll
            for (int i = 0; i < KP; ++i)
              if (i == l8 + 8 * o) so = rs[i];
            dot[o] = fmaf(fin * rcf, cnt[so], dot[o]);
          }
        }
#pragma unroll
        for (int k = 0; k < CPL; ++k) sum[k] *= fin;
      }
      // outputs
#pragma unroll
      for (int o = 0; o < NO; ++o) {
        const int i = l8 + 8 * o;
        dot_out[static_cast<int64_t>(t) * KP + i] = i < kk ? dot[o] : 0.f;
      }
      if (REV) {
#pragma unroll
        for (int k = 0; k < CPL; ++k) sum[k] += cur.sum.e[k];
        const int64_t at = n * a.sum_stride + static_cast<int64_t>(h) * a.dh + col0 + CPL * l8;
        if (a.sum_bf16) store_vals<CPL, bf16_t>(static_cast<bf16_t*>(a.sum_out) + at, sum);
        else store_vals<CPL, float>(static_cast<float*>(a.sum_out) + at, sum);
      }
    }

    // the written rows' new values (no other group writes them, so they can be summed before the reads are done):
    // the old row faded by the chunk (as mu; by itself where the slab is rescaled; none of it where a reset empties the
    // slab, chosen and not multiplied by zero, which would keep an infinity's NaN), the slot's first writer and its
    // later ones from the chain.  Group g takes records g + 64 k; null records (row M) write nothing
    const float mu_all = mu * pw[L];
    // the slab takes the scale in, mu restarts at 1 (the same in every lane: a branch around it costs a chunk nothing)
    const bool fold = __builtin_amdgcn_readfirstlane(rmask != 0 || !(mu_all >= kMuFloor));
    const float inv_mu = fold ? 1.f : fast_rcp(mu_all);
    const unsigned char* gext = chains + static_cast<int64_t>(c) * chain_stride(KP) + 16 + 8 * kChunk * KP;
    auto ext_at = [&](int e) {
      return 8 * e + 8 <= XS ? reinterpret_cast<const uint2*>(s_ext)[e] : reinterpret_cast<const uint2*>(gext)[e];
    };
    auto row_of = [&](int q) { return lds_seg<CPL>(&s_wv[(q & 63) * CW + CPL * l8]); };
    Seg<CPL> x[KP];
    int slot_of[KP], own_slot[NO];
    float own_cnt[NO];
#pragma unroll
    for (int k0 = 0; k0 < KP; k0 += 8) {
      uint2 wr[8];
#pragma unroll
      for (int j = 0; j < 8; j += 2) {
        const uint4 r2 = *reinterpret_cast<const uint4*>(&s_rec[g * KP + k0 + j]);
        wr[j] = make_uint2(r2.x, r2.y);
        wr[j + 1] = make_uint2(r2.z, r2.w);
      }
      Seg<CPL> vq[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        slot_of[k0 + j] = static_cast<int>(wr[j].x & 0xffffu);
        x[k0 + j] = lds_seg<CPL>(&A[slot_of[k0 + j] * CW + CPL * l8]);
        vq[j] = row_of(wr[j].x >> 16);
      }
      const uint2 ow = cur.own_w[k0 / 8];   // the lane's count: record k0 + l8
      own_slot[k0 / 8] = static_cast<int>(ow.x & 0xffffu);
      float cold = cnt[own_slot[k0 / 8]];
      if (fold) {
        cold = rmask ? 0.f : cold * mu_all;
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int k = 0; k < CPL; ++k) x[k0 + j].v[k] = rmask ? 0.f : x[k0 + j].v[k] * mu_all;
      }
      float dcc = __uint_as_float(ow.y & 0x7fffffffu) * s_wc[(ow.x >> 16) & 63u];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float dc = __uint_as_float(wr[j].y & 0x7fffffffu) * inv_mu;
#pragma unroll
        for (int k = 0; k < CPL; ++k) x[k0 + j].v[k] = fmaf(dc, vq[j].v[k], x[k0 + j].v[k]);
      }
      // the later writers of two records at a time, the next entries loaded ahead: a chain costs one LDS round trip a
      // writer, and the two records' overlap
#pragma unroll
      for (int j = 0; j < 8; j += 2) {
        bool l0 = wr[j].y >> 31, l1 = wr[j + 1].y >> 31;
        if (l0 || l1) {
          int e0 = wr[j].x >> 22, e1 = wr[j + 1].x >> 22;
          uint2 t0 = ext_at(min(e0, kChunk * KP - 1)), t1 = ext_at(min(e1, kChunk * KP - 1));
          do {
            const Seg<CPL> v0 = row_of(t0.y), v1 = row_of(t1.y);
            const float w0 = s_wc[t0.y & 63u], w1 = s_wc[t1.y & 63u];
            const uint2 n0 = ext_at(min(++e0, kChunk * KP - 1)), n1 = ext_at(min(++e1, kChunk * KP - 1));
            const float c0 = __uint_as_float(t0.x), c1 = __uint_as_float(t1.x);
#pragma unroll
            for (int k = 0; k < CPL; ++k) {
              x[k0 + j].v[k] = l0 ? fmaf(c0 * inv_mu, v0.v[k], x[k0 + j].v[k]) : x[k0 + j].v[k];
              x[k0 + j + 1].v[k] = l1 ? fmaf(c1 * inv_mu, v1.v[k], x[k0 + j + 1].v[k]) : x[k0 + j + 1].v[k];
            }
            dcc = l0 && l8 == j ? fmaf(c0, w0, dcc) : dcc;
            dcc = l1 && l8 == j + 1 ? fmaf(c1, w1, dcc) : dcc;
            l0 = l0 && !(t0.y >> 31);
            l1 = l1 && !(t1.y >> 31);
            t0 = n0;
            t1 = n1;
          } while (l0 || l1);
        }
      }
      own_cnt[k0 / 8] = fmaf(dcc, inv_mu, cold);
    }
    lds_barrier();   // every read of the slab and of the staged chunk is done

    if (fold) {
      for (int i = tid; i < M * CW; i += kGradScanThreads) A[i] = rmask ? 0.f : A[i] * mu_all;
      for (int i = tid; i < M; i += kGradScanThreads) cnt[i] = rmask ? 0.f : cnt[i] * mu_all;
      lds_barrier();
    }
#pragma unroll
    for (int j = 0; j < KP; ++j)
      if (slot_of[j] != M) lds_seg_store<CPL>(&A[slot_of[j] * CW + CPL * l8], x[j]);
#pragma unroll
    for (int o = 0; o < NO; ++o)
      if (own_slot[o] != M) cnt[own_slot[o]] = own_cnt[o];
    mu = fold ? 1.f : mu_all;
    if (more) {
      stage(nxt, g < ChunkSpan<REV>(c + 1, T, a.n_chunks).L);
      cur = nxt;
    }
    lds_barrier();
  }
}

// ---------------------------------------------------------------------------------------------------------------
// addr_grad_kernel: softmax, gate, address normalisation and sub-key products backward, one wave per (token, head,
// address set) at a time, lane e = address element e (d_a = 2 * HALF <= 64); lane j < KP also holds pick j for the
// softmax and gate math, whose per-pick results reach every lane by v_readlane.  Block (token block, head, set) of W
// waves (4 per SIMD: their memory round trips overlap); wave w takes tokens n_begin + w + W i.
//   read set:  x_j = tau sv_j, wr = softmax(x):          dx_j = wr_j (dwr_j - P), P = sum_j wr_j dwr_j
//   write set: ww = softmax(tau sv) * g:                 dp_j = g dww_j, dx_j = p_j (dp_j - sum p dp),
//                                                        dg = sum_j p_j dww_j, dlogit = dg g (1 - g)
//   both:      dsv_j = tau dx_j, dtau += sum_j sv_j dx_j; sv_j = (v1[i1_j] + v2[i2_j]) / 2 with v = <u, k^>:
//              du += dsv_j / 2 k^[i_j], dk^[i_j] += dsv_j / 2 u; u = z / max(|z|, 1e-12):
//              dz = (du - u <u, du>) / |z| (du / 1e-12 below the floor); z = kz + addr_b
// Per block: partial sums of dtau, the gate bias, addr_b, lam dL/dlam (float64) and the unit sub-key gradient (one
// copy per wave in LDS, summed in wave order: no atomics, a fixed order).
constexpr int kAddrGradWaveTokens = 16;   // tokens per wave
// waves per block at most (4 per SIMD; the kernel needs well under 128 registers)
__host__ __device__ constexpr int addr_grad_max_waves(int) { return 16; }

struct AddrGradArgs {
  const void* kz;
  int64_t kz_stride;
  const void* qz;
  int64_t qz_stride;
  const void* gl;            // gate logit rows or nullptr (no gate)
  int64_t g_stride;
  const float* keys[2];      // raw sub-keys [H][n_sub][HALF]
  const float* addr_b;       // [H][d_a] or nullptr
  const float* log_scale;    // [H]
  const float* gate_bias;    // [H] or nullptr
  const int32_t* slot[2];    // [B][H][T][KP]: write, read
  const float* wt[2];
  const float* score[2];
  const float* dot[2];       // [CG][B][H][T][KP] per-pick gradient partials: dww, dwr
  int n_cg;
  void* dz[2];               // rows of H * d_a: d kz, d qz (float32; bfloat16 with out_bf16, as dgl)
  int64_t dz_stride[2];
  void* dgl;                 // rows of H or nullptr
  int64_t dgl_stride;
  int out_bf16;
  float* part_f;             // [n_blk][2][H][2 + d_a]: dtau, d gate bias, d addr_b
  double* part_d;            // [n_blk][2][H]: lam dL/dlam
  float* part_k;             // [n_blk][2][H][2][n_sub][HALF]: d unit sub-keys
  int B, T, H, n_sub, kk;
  int set0;                  // the first address set (grid z covers set0 .. set0 + gridDim.z - 1)
  int wave_tokens;           // tokens per wave (addr_grad_tile_kernel: a multiple of its 32-token tile)
};


// an input gradient in the caller's type
__device__ __forceinline__ void store_grad(void* p, int64_t i, float v, int as_bf16) {
  if (as_bf16) static_cast<bf16_t*>(p)[i] = from_f32<bf16_t>(v);
  else static_cast<float*>(p)[i] = v;
}

__device__ __forceinline__ float lane_f(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// sum over aligned groups of 16 lanes (the rows of the wave), by DPP
__device__ __forceinline__ float sum16(float v) {
  v = sum8(v);
  return v + dpp_f<0x140>(v);   // row_mirror: lane i and lane 15 - i hold the two 8-lane sums
}

// sum over the 64 lanes (every lane active): the rows by DPP, then the four row sums read out of lanes 0, 16, 32, 48
__device__ __forceinline__ float wave_sum(float v) {
  const float s = sum16(v);
  return (lane_f(s, 0) + lane_f(s, 16)) + (lane_f(s, 32) + lane_f(s, 48));
}

// sum over the lane's half of the address (lanes [0, HALF) or [HALF, 2 HALF))
template <int HALF>
__device__ __forceinline__ float half_sum(float v, int e) {
  if constexpr (HALF == 32) {   // rows 0 + 1 and 2 + 3
    const float s = sum16(v);
    const float s0 = lane_f(s, 0) + lane_f(s, 16);
    const float s1 = lane_f(s, 32) + lane_f(s, 48);
    return e < 32 ? s0 : s1;
  } else if constexpr (HALF == 16) {
    return sum16(v);
  } else if constexpr (HALF == 8) {
    return sum8(v);
  } else if constexpr ((HALF & (HALF - 1)) == 0) {   // aligned groups of HALF lanes
#pragma unroll
    for (int off = 1; off < HALF; off <<= 1) v += __shfl_xor(v, off);
    return v;
  } else {
    const float s1 = wave_sum(e < HALF ? v : 0.f);
    const float s2 = wave_sum(e >= HALF && e < 2 * HALF ? v : 0.f);
    return e < HALF ? s1 : s2;
  }
}

// LDS of addr_grad_kernel for W waves: wave partials of lam dL/dlam (float64), unit sub-keys, one sub-key gradient
// copy and one partial record per wave
__host__ __device__ constexpr size_t addr_grad_lds(int n_sub, int half, int W) {
  return sizeof(double) * W + sizeof(float) * (2 * static_cast<size_t>(n_sub) * half * (1 + W) + W * (2 * half + 2));
}

// sum over lanes [0, KP) (aligned groups of KP lanes; KP a power of two)
template <int KP>
__device__ __forceinline__ float pick_sum(float v) {
  if constexpr (KP == 8) {
    return sum8(v);
  } else if constexpr (KP == 16) {
    return sum16(v);
  } else {
#pragma unroll
    for (int off = 1; off < KP; off <<= 1) v += __shfl_xor(v, off);
    return v;
  }
}


// one block of addr_grad_kernel, on addr_grad_lds(n_sub, HALF, its waves) bytes of LDS
template <int HALF, int KP, typename InT>
__device__ __forceinline__ void addr_grad_block(const AddrGradArgs& a, unsigned char* albuf) {
  constexpr int DA = 2 * HALF;
  const int W = blockDim.x >> 6;
  const int n_sub = a.n_sub;
  const int KS = 2 * n_sub * HALF;                                // sub-key values of both halves
  double* redd = reinterpret_cast<double*>(albuf);                // [W]
  float* kn = reinterpret_cast<float*>(albuf + sizeof(double) * W);   // [2][n_sub][HALF] unit sub-keys
  float* dk = kn + KS;                                            // [W][2][n_sub][HALF] their gradient per wave
  float* red = dk + W * KS;                                       // [W][DA + 2] wave partials
  const int h = blockIdx.y;
  const int set = a.set0 + blockIdx.z;   // 0: write keys, 1: read queries
  const int tid = threadIdx.x;
  const int w = tid >> 6;
  const int e = tid & 63;       // address element; lanes e < KP also hold pick e
  const int kk = a.kk;
  if constexpr ((HALF & (HALF - 1)) == 0) {   // unit sub-keys: one row per aligned group of HALF lanes, all waves
    for (int i0 = w * 64; i0 < KS; i0 += blockDim.x) {   // wave-uniform bound: every lane takes the lane sums
      const int i = i0 + e;
      const int r = i / HALF;
      const int part = r >= n_sub;
      const float v = i < KS ? a.keys[part][(static_cast<int64_t>(h) * n_sub + (r - part * n_sub)) * HALF + i % HALF]
                             : 0.f;
      const float nrm = fmaxf(sqrtf(half_sum<HALF>(v * v, e)), 1e-12f);
      if (i < KS) kn[i] = v / nrm;
    }
  } else {
    for (int r = tid; r < 2 * n_sub; r += blockDim.x) {
      const int part = r >= n_sub;
      const float* src = a.keys[part] + (static_cast<int64_t>(h) * n_sub + (r - part * n_sub)) * HALF;
      float ss = 0.f;
      for (int d = 0; d < HALF; ++d) ss = fmaf(src[d], src[d], ss);
      const float nrm = fmaxf(sqrtf(ss), 1e-12f);
      for (int d = 0; d < HALF; ++d) kn[r * HALF + d] = src[d] / nrm;
    }
  }
  for (int i = tid; i < W * KS; i += blockDim.x) dk[i] = 0.f;
  __syncthreads();
  float* dkw = dk + w * KS;   // this wave's copy: within a wave the lanes of one pick touch distinct entries
  const float tau = expf(a.log_scale[h]);
  const float ab = (e < DA && a.addr_b) ? a.addr_b[h * DA + e] : 0.f;
  const float gb = a.gate_bias ? a.gate_bias[h] : 0.f;
  const int hf = e >= HALF;               // the lane's half
  const int ec = e - hf * HALF;           // column within the half
  // slot -> (i1, i2) = (s / n_sub, s % n_sub) by a multiply-high: exact for s < 2^16, n_sub <= 256
  const uint32_t magic = n_sub > 1 ? 0xFFFFFFFFu / static_cast<uint32_t>(n_sub) + 1u : 0u;
  const InT* zb = static_cast<const InT*>(set == 0 ? a.kz : a.qz);
  const int64_t zs = set == 0 ? a.kz_stride : a.qz_stride;
  const bool gated = set == 0 && a.gl;
  const int32_t* slot = a.slot[set];
  const float* wtp = a.wt[set];
  const float* scp = a.score[set];
  const float* dotp = a.dot[set];
  void* dzp = a.dz[set];
  const int64_t dzs = a.dz_stride[set];
  const bool pl = e < kk;                 // the lane holds a live pick
  float acc_tau = 0.f, acc_gb = 0.f, acc_ab = 0.f;
  double acc_lam = 0.0;
  const int64_t N = static_cast<int64_t>(a.B) * a.T;
  const int64_t cg_stride = N * a.H * KP;
  int64_t n = static_cast<int64_t>(blockIdx.x) * W * a.wave_tokens + w;
  int b = static_cast<int>(n / a.T);
  int t = static_cast<int>(n - static_cast<int64_t>(b) * a.T);
  // one token's loads, issued a token ahead: unconditional, at indexes clamped into the arrays (masked after use)
  struct TokIn {
    InT z, gl;
    int sl;
    float sv, wt, d0, d1;
  };
  const int ez = (DA == 64 || e < DA) ? e : 0;
  const int ep = pl ? e : 0;
  auto load = [&](int64_t nn, int bb, int tt) {
    TokIn x;
    const int64_t prow = ((static_cast<int64_t>(bb) * a.H + h) * a.T + tt) * KP + ep;
    x.z = zb[nn * zs + static_cast<int64_t>(h) * DA + ez];
    x.gl = gated ? static_cast<const InT*>(a.gl)[nn * a.g_stride + h] : zb[0];
    x.sl = slot[prow];
    x.sv = scp[prow];
    x.wt = wtp[prow];
    x.d0 = dotp[prow];
    x.d1 = a.n_cg > 1 ? dotp[cg_stride + prow] : 0.f;
    return x;
  };
  TokIn cur = load(n < N ? n : 0, n < N ? b : 0, n < N ? t : 0);
  for (int i = 0; i < a.wave_tokens; ++i) {
    if (n >= N) break;   // wave-uniform
    // the next token (W positions on) and its loads
    const int64_t n2 = n + W;
    int b2 = b, t2 = t + W;
    while (t2 >= a.T) {
      t2 -= a.T;
      ++b2;
    }
    TokIn nxt = cur;
    if (i + 1 < a.wave_tokens && n2 < N) nxt = load(n2, b2, t2);
    const int64_t prow = ((static_cast<int64_t>(b) * a.H + h) * a.T + t) * KP;
    const float z = (DA == 64 || e < DA) ? to_f32(cur.z) + ab : 0.f;
    const float glv = gated ? to_f32(cur.gl) : 0.f;
    int sl = pl ? cur.sl : 0;
    sl = (sl >= 0 && sl < n_sub * n_sub) ? sl : 0;
    const float sv = pl ? cur.sv : 0.f;
    const float wt = pl ? cur.wt : 0.f;
    float dw = pl ? cur.d0 + cur.d1 : 0.f;
    for (int c = 2; c < a.n_cg; ++c) dw += pl ? dotp[c * cg_stride + prow + e] : 0.f;
    // softmax (and gate) backward, pick e on lane e
    float dx;
    if (set == 1) {   // read: softmax
      const float P = pick_sum<KP>(wt * dw);
      dx = wt * (dw - P);
      acc_lam += static_cast<double>(t) * static_cast<double>(P);
    } else {          // write: gated softmax
      const float Q = pick_sum<KP>(wt * dw);
      acc_lam -= static_cast<double>(t + 1) * static_cast<double>(Q);
      const float x0 = lane_f(sv, 0) * tau;
      float pj = pl ? __expf(sv * tau - x0) : 0.f;
      pj *= fast_rcp(pick_sum<KP>(pj));
      const float gt = gated ? fast_rcp(1.f + __expf(-(glv + gb))) : 1.f;
      const float S = pick_sum<KP>(pj * gt * dw);
      const float dg = pick_sum<KP>(pj * dw);
      dx = pj * (gt * dw - S);
      if (gated) {
        const float dlogit = dg * gt * (1.f - gt);
        if (e == 0 && a.dgl) store_grad(a.dgl, n * a.dgl_stride + h, dlogit, a.out_bf16);
        acc_gb += e == 0 ? dlogit : 0.f;
      }
    }
    if (!pl) dx = 0.f;
    acc_tau = fmaf(sv, dx, acc_tau);        // per lane (pick), summed over lanes at the end
    const float hs = 0.5f * tau * dx;        // d sv / 2 of pick e
    const int i1 = n_sub > 1 ? static_cast<int>(__umulhi(static_cast<uint32_t>(sl), magic)) : sl;
    const int i2 = sl - i1 * n_sub;
    const float z2 = z * z;
    const float nz = __builtin_amdgcn_sqrtf(half_sum<HALF>(z2, e));
    const float inz = fast_rcp(fmaxf(nz, 1e-12f));
    const float u = z * inz;
    // pick j: du += hs_j k^[i_j], dk^[i_j] += hs_j u.  Both row offsets are read out of pick lane j and the lane's
    // half selects one (no branch); picks sharing a row add up in pick order
    const int off1 = i1 * HALF;
    const int off2 = (n_sub + i2) * HALF;
    float du = 0.f;
#pragma unroll
    for (int j = 0; j < KP; ++j) {
      if (j >= kk) break;   // uniform
      const float hj = lane_f(hs, j);
      const int o1 = __builtin_amdgcn_readlane(off1, j);
      const int o2 = __builtin_amdgcn_readlane(off2, j);
      const int o = (hf ? o2 : o1) + ec;
      if (DA == 64 || e < DA) {
        du = fmaf(hj, kn[o], du);
        dkw[o] += hj * u;
      }
    }
    const float ud = half_sum<HALF>(u * du, e);
    const float dz = nz > 1e-12f ? (du - u * ud) * inz : du * 1e12f;
    if (e < DA) store_grad(dzp, n * dzs + static_cast<int64_t>(h) * DA + e, dz, a.out_bf16);
    acc_ab += dz;
    cur = nxt;
    n = n2;
    b = b2;
    t = t2;
  }
  acc_tau = wave_sum(acc_tau);   // the picks' lanes, in a fixed order
  // block sums in a fixed order: waves -> LDS -> threads
  if (e < DA) red[w * (DA + 2) + e] = acc_ab;
  if (e == 0) {
    red[w * (DA + 2) + DA] = acc_tau;
    red[w * (DA + 2) + DA + 1] = acc_gb;
    redd[w] = acc_lam;
  }
  __syncthreads();
  const int64_t pid = (static_cast<int64_t>(blockIdx.x) * gridDim.z + blockIdx.z) * a.H + h;
  for (int c = tid; c < DA + 2; c += blockDim.x) {
    float s = 0.f;
    for (int q = 0; q < W; ++q) s += red[q * (DA + 2) + c];
    // record order: dtau, d gate bias, d addr_b[DA]
    const int f = c == DA ? 0 : c == DA + 1 ? 1 : 2 + c;
    a.part_f[pid * (2 + DA) + f] = s;
  }
  if (tid == 0) {
    double s = 0.0;
    for (int q = 0; q < W; ++q) s += redd[q];
    a.part_d[pid] = s;
  }
  for (int i = tid; i < KS; i += blockDim.x) {
    float s = 0.f;
    for (int q = 0; q < W; ++q) s += dk[q * KS + i];
    a.part_k[pid * KS + i] = s;
  }
}

template <int HALF, int KP, typename InT>
__global__ void __launch_bounds__(64 * addr_grad_max_waves(KP)) addr_grad_kernel(AddrGradArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char agbuf[];
  addr_grad_block<HALF, KP, InT>(a, agbuf);
}

// ---------------------------------------------------------------------------------------------------------------
// addr_grad_tile_kernel: the same gradients for n_sub <= 64, 32 tokens of one (head, address set) at a time on the
// matrix cores.  Per tile a wave
//   picks   holds KP lanes per token (64 / KP tokens side by side, so every lane has a pick): softmax and gate
//           backward by DPP over the token's lanes, then g_j = dsv_j / 2 added into the token's row of G, its
//           sparse gradient by unit sub-key (LDS, [32 tokens][both halves' sub-keys]; picks in pick order)
//   du      = G K^ (v_mfma_f32_32x32x2f32: rows tokens, columns address elements)
//   dz      from du, u and |z|, held in the product's own layout: lane l keeps column l % 32 of 16 tokens, so the
//           sums over an address half are sums over lanes of a half-wave
//   dk^    += G^T U (the products' tokens in the order U's registers hold them)
// Everything stays float32 (the products are fused multiply-adds in float32).  addr_grad_kernel does the same one
// token at a time, one lane per address element: per token 8 dependent LDS read-modify-writes for dk^, 24 readlanes
// and the pick math on 8 of 64 lanes.  B=8, T=2048, 12 heads, k=8, bfloat16: 218 us so, 117 here on the same two partials
// of a pick's dot, 130 on the three that it has with chunk_grad_kernel's; the table layer's (B=4, T=1024, one head, 64
// sub-keys, k=16, float32): 50 and 33 us.  What bounds it: 176 MB in and out (36 us at a
// copy's rate; 226 with row gradients in float32), and the latency of a tile's chain (loads, k LDS additions, products) with two waves per SIMD: the
// kernel takes 256 registers (with two blocks of sub-keys 10 to 73 of them spilled), and at three waves (168, 73 of them
// spilled with one) it took 141 us.
// Sub-keys past n_sub, columns past the address and tokens past the end are zero rows and columns of the tiles.
// The products run over every sub-key and 32 tokens, and 0 times an infinity is NaN: a block that meets an address or a
// sub-key that is not finite does all its tokens again one at a time (addr_grad_block), so that it reaches no more than
// its own picks.
// Waves per block 4; tiles per wave chosen by addr_tiles (enough blocks for the chip first, then longer waves, since
// every wave loads the head's sub-keys and leaves a partial sum).
constexpr int kAddrTile = 32;
constexpr int kAddrTileWaves = 4;   // (the waves' flags at the kernel's end are four)

// sum over the 32 lanes of the lane's half-wave
__device__ __forceinline__ float sum32(float v) {
  v = sum16(v);
  const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
}

// orders the LDS accesses of a wave's lanes among themselves (the hardware runs a wave's LDS operations in order)
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// sum over the columns of the lane's address half: columns 0 .. HALF - 1 of a half-wave with HALF > 16 (a tile per
// half), else columns [0, HALF) or [HALF, 2 HALF); columns past them hold zero
template <int HALF>
__device__ __forceinline__ float col_sum(float v, int col) {
  if constexpr (HALF > 16) {
    return sum32(v);
  } else if constexpr (HALF == 16) {
    return sum16(v);
  } else if constexpr (HALF == 8) {
    return sum8(v);
  } else {
    const float s1 = sum32(col < HALF ? v : 0.f);
    const float s2 = sum32(col >= HALF ? v : 0.f);
    return col < HALF ? s1 : s2;
  }
}

// LDS of one addr_grad_tile block: the waves' G tiles and the unit sub-keys, in the same bytes at the end their dk^ and partial records
__host__ __device__ constexpr int addr_tile_pitch(int nsb) { return 64 * nsb + 4; }
__host__ __device__ constexpr size_t addr_tile_lds(int n_sub, int half, int nsb) {
  const size_t g = sizeof(float) * (kAddrTileWaves * kAddrTile * addr_tile_pitch(nsb) + 64 * nsb * 32);
  const size_t d = sizeof(float) * kAddrTileWaves * 2 * static_cast<size_t>(n_sub) * half;
  const size_t t = (g > d ? g : d) + kAddrTileWaves * (sizeof(double) + sizeof(float) * (2 * half + 2));
  const size_t o = (addr_grad_lds(n_sub, half, kAddrTileWaves) + 7) / 8 * 8;   // one token at a time
  return t > o ? t : o;
}

__device__ __forceinline__ bool finite_f32(float v) { return fabsf(v) <= 3.402823466e38f; }

template <int HALF, int NSB, int KP, typename InT>
__global__ void __launch_bounds__(64 * kAddrTileWaves, 2) addr_grad_tile_kernel(AddrGradArgs a) {
  constexpr int DA = 2 * HALF;
  constexpr int NT = HALF > 16 ? 2 : 1;          // column tiles: one per half, or both halves in one
  constexpr int SB = 32 * NSB;                   // G columns of one half
  constexpr int GP = addr_tile_pitch(NSB);
  constexpr int TPI = 64 / KP;                   // tokens per pick step
  constexpr int NIT = kAddrTile / TPI;
  extern __shared__ __attribute__((aligned(16))) unsigned char albuf[];
  const int n_sub = a.n_sub;
  const int KS = 2 * n_sub * HALF;
  const int h = blockIdx.y;
  const int set = a.set0 + blockIdx.z;   // 0: write keys, 1: read queries
  const int tid = threadIdx.x;
  const int w = tid >> 6;
  const int lane = tid & 63;
  const int col = lane & 31;             // column of a tile; in G's products also a token or a sub-key
  const int hw = lane >> 5;
  const int pj = lane & (KP - 1);        // the lane's pick in the pick steps
  const int kk = a.kk;
  float* G = reinterpret_cast<float*>(albuf) + w * kAddrTile * GP;

  // the unit sub-keys, [half][sub-key][column of its tile]: zero past n_sub and, with both halves in one tile, in the
  // other half's columns
  float* kn = reinterpret_cast<float*>(albuf) + kAddrTileWaves * kAddrTile * GP;
  __shared__ int s_odd[kAddrTileWaves];   // whether the wave met an address or a sub-key that is not finite
  bool fin = true;
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const float* keys = a.keys[p] + static_cast<int64_t>(h) * n_sub * HALF;
    const int c = NT == 2 ? col : col - p * HALF;
    const bool own = c >= 0 && c < HALF;
    for (int i0 = 2 * w; i0 < SB; i0 += 2 * kAddrTileWaves) {   // two rows a wave: one per half-wave
      const int i = i0 + hw;
      const float v = own && i < n_sub ? keys[i * HALF + c] : 0.f;
      const float nrm = fmaxf(sqrtf(col_sum<HALF>(v * v, col)), 1e-12f);
      const float kv = v / nrm;
      fin = fin && finite_f32(kv);
      kn[(p * SB + i) * 32 + col] = kv;
    }
  }
  __syncthreads();
  const float tau = expf(a.log_scale[h]);
  float ab[NT];
#pragma unroll
  for (int p = 0; p < NT; ++p) {
    const int e = p * HALF + col;
    ab[p] = a.addr_b && (NT == 2 ? col < HALF : col < DA) ? a.addr_b[h * DA + e] : 0.f;
  }
  const float gb = a.gate_bias ? a.gate_bias[h] : 0.f;
  // slot -> (i1, i2) = (s / n_sub, s % n_sub) by a multiply-high: exact for s < 2^16, n_sub <= 256
  const uint32_t magic = n_sub > 1 ? 0xFFFFFFFFu / static_cast<uint32_t>(n_sub) + 1u : 0u;
  const InT* zb = static_cast<const InT*>(set == 0 ? a.kz : a.qz) + static_cast<int64_t>(h) * DA;
  const int zs = static_cast<int>(set == 0 ? a.kz_stride : a.qz_stride);   // below 2^25 (the launcher's rule)
  const bool gated = set == 0 && a.gl;
  const int32_t* slot = a.slot[set];
  const float* wtp = a.wt[set];
  const float* scp = a.score[set];
  const float* dotp = a.dot[set];
  const int dzs = static_cast<int>(a.dz_stride[set]);
  const bool live_col = NT == 2 ? col < HALF : col < DA;
  const int64_t N = static_cast<int64_t>(a.B) * a.T;   // below 2^31: each token has picks of 4 * 32 bytes and more
  const int64_t cg_stride = N * a.H * KP;
  float acc_ab[NT];
  double acc_lam = 0.0, acc_tau = 0.0, acc_gb = 0.0;
  floatx16 dk[2][NSB];
#pragma unroll
  for (int p = 0; p < NT; ++p) acc_ab[p] = 0.f;
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int q = 0; q < NSB; ++q)
#pragma unroll
      for (int r = 0; r < 16; ++r) dk[p][q][r] = 0.f;

  int64_t n0 = (static_cast<int64_t>(blockIdx.x) * kAddrTileWaves + w) * a.wave_tokens;
  for (int i = 0; i < a.wave_tokens && n0 < N; i += kAddrTile, n0 += kAddrTile) {   // wave-uniform
    // loads: unconditional, a missing token reads token 0 and a dead pick the token's first (masked after use)
    int slr[NIT], tr[NIT];
    float svr[NIT], wtr[NIT], dwr[NIT];
    InT glr[NIT];
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const int64_t nn = n0 + it * TPI + lane / KP;
      const uint32_t n = nn < N ? static_cast<uint32_t>(nn) : 0u;
      const uint32_t b = n / static_cast<uint32_t>(a.T);
      const uint32_t t = n - b * static_cast<uint32_t>(a.T);
      const int64_t e = ((static_cast<int64_t>(b) * a.H + h) * a.T + t) * KP + (pj < kk ? pj : 0);
      tr[it] = static_cast<int>(t);
      slr[it] = slot[e];
      svr[it] = scp[e];
      wtr[it] = wtp[e];
      // up to three partials (a head of 64 columns) in straight code: their loads issue with the others
      const float d1 = dotp[(a.n_cg > 1 ? cg_stride : 0) + e], d2 = dotp[(a.n_cg > 2 ? 2 * cg_stride : 0) + e];
      dwr[it] = dotp[e] + (a.n_cg > 1 ? d1 : 0.f) + (a.n_cg > 2 ? d2 : 0.f);
      for (int c = 3; c < a.n_cg; ++c) dwr[it] += dotp[c * cg_stride + e];
      glr[it] = gated ? static_cast<const InT*>(a.gl)[n * a.g_stride + h] : zb[0];
    }
    const InT* zt = zb + n0 * zs;   // the tile's rows: offsets from here in 32 bits
    const int left = static_cast<int>(N - n0 < kAddrTile ? N - n0 : kAddrTile);
    InT zr[NT][16];
#pragma unroll
    for (int p = 0; p < NT; ++p)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 8 * (r / 4) + 4 * hw + r % 4;
        zr[p][r] = zt[(row < left ? row : 0) * zs + (live_col ? p * HALF + col : 0)];
      }
    const int64_t dz0 = n0 * a.dz_stride[set] + static_cast<int64_t>(h) * DA;   // the tile's first output value
    float* dzt = static_cast<float*>(a.dz[set]) + dz0;
    bf16_t* dzb = static_cast<bf16_t*>(a.dz[set]) + dz0;
    // G to zero, then the picks' gradients
#pragma unroll
    for (int k = 0; k < (kAddrTile * GP + 255) / 256; ++k) {
      const int at = 4 * (lane + 64 * k);
      if (at < kAddrTile * GP) *reinterpret_cast<float4*>(&G[at]) = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    float hs[NIT];
    int g1[NIT], g2[NIT];
#pragma unroll
    for (int it = 0; it < NIT; ++it) {
      const bool valid = n0 + it * TPI + lane / KP < N;
      const bool pl = valid && pj < kk;
      int sl = pl ? slr[it] : 0;
      sl = (sl >= 0 && sl < n_sub * n_sub) ? sl : 0;
      const float sv = pl ? svr[it] : 0.f;
      const float wt = pl ? wtr[it] : 0.f;
      const float dw = pl ? dwr[it] : 0.f;
      const float P = pick_sum<KP>(wt * dw);
      const float sv0 = __shfl(sv, lane & ~(KP - 1));   // the token's best score
      float dx;
      if (set == 1) {   // read: softmax
        dx = wt * (dw - P);
        if (pj == 0) acc_lam += static_cast<double>(tr[it]) * static_cast<double>(P);
      } else {          // write: gated softmax
        if (pj == 0) acc_lam -= static_cast<double>(tr[it] + 1) * static_cast<double>(P);
        float pr = pl ? __expf(sv * tau - sv0 * tau) : 0.f;
        const float ps = pick_sum<KP>(pr);
        pr *= fast_rcp(valid ? ps : 1.f);
        const float gt = gated ? fast_rcp(1.f + __expf(-(to_f32(glr[it]) + gb))) : 1.f;
        const float S = pick_sum<KP>(pr * gt * dw);
        const float dg = pick_sum<KP>(pr * dw);
        dx = pr * (gt * dw - S);
        if (gated && valid && pj == 0) {
          const float dlogit = dg * gt * (1.f - gt);
          if (a.dgl) store_grad(a.dgl, (n0 + it * TPI + lane / KP) * a.dgl_stride + h, dlogit, a.out_bf16);
          acc_gb += dlogit;
        }
      }
      if (!pl) dx = 0.f;
      // a token's dx sum to zero, so its scores count from the best one: small terms instead of large ones that cancel
      acc_tau += static_cast<double>((sv - sv0) * dx);
      hs[it] = 0.5f * tau * dx;
      const int i1 = n_sub > 1 ? static_cast<int>(__umulhi(static_cast<uint32_t>(sl), magic)) : sl;
      const int row = (it * TPI + lane / KP) * GP;
      g1[it] = row + i1;
      g2[it] = row + SB + (sl - i1 * n_sub);
    }
    wave_lds_fence();
#pragma unroll
    for (int j = 0; j < KP; ++j) {
      if (j >= kk) break;   // uniform
      if (pj == j) {        // one lane per token: picks of a token that share a sub-key add up in pick order
        float x1[NIT], x2[NIT];
#pragma unroll
        for (int it = 0; it < NIT; ++it) {
          x1[it] = G[g1[it]];
          x2[it] = G[g2[it]];
        }
#pragma unroll
        for (int it = 0; it < NIT; ++it) {
          G[g1[it]] = x1[it] + hs[it];
          G[g2[it]] = x2[it] + hs[it];
        }
      }
      wave_lds_fence();
    }
#pragma unroll
    for (int p = 0; p < NT; ++p) {
      // du: rows tokens, columns address elements; lane l's sub-keys at step s are 16 (l / 32) + s of each block
      floatx16 du;
#pragma unroll
      for (int r = 0; r < 16; ++r) du[r] = 0.f;
#pragma unroll
      for (int pp = 0; pp < 2; ++pp) {
        if (NT == 2 && pp != p) continue;
#pragma unroll
        for (int q = 0; q < NSB; ++q)
#pragma unroll
          for (int s4 = 0; s4 < 4; ++s4) {
            const float4 g4 = *reinterpret_cast<const float4*>(&G[col * GP + pp * SB + 32 * q + 16 * hw + 4 * s4]);
            const float* kr = &kn[(pp * SB + 32 * q + 16 * hw + 4 * s4) * 32 + col];
            du = __builtin_amdgcn_mfma_f32_32x32x2f32(g4.x, kr[0], du, 0, 0, 0);
            du = __builtin_amdgcn_mfma_f32_32x32x2f32(g4.y, kr[32], du, 0, 0, 0);
            du = __builtin_amdgcn_mfma_f32_32x32x2f32(g4.z, kr[64], du, 0, 0, 0);
            du = __builtin_amdgcn_mfma_f32_32x32x2f32(g4.w, kr[96], du, 0, 0, 0);
          }
      }
      float u[16], inz[16], nz[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const bool live = live_col && 8 * (r / 4) + 4 * hw + r % 4 < left;
        const float z = live ? to_f32(zr[p][r]) + ab[p] : 0.f;
        nz[r] = __builtin_amdgcn_sqrtf(col_sum<HALF>(z * z, col));
        inz[r] = fast_rcp(fmaxf(nz[r], 1e-12f));
        u[r] = z * inz[r];
      }
      // dk^: rows sub-keys, columns address elements; register r's two tokens are the step's two
#pragma unroll
      for (int pp = 0; pp < 2; ++pp) {
        if (NT == 2 && pp != p) continue;
#pragma unroll
        for (int q = 0; q < NSB; ++q)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float gt = G[(8 * (r / 4) + 4 * hw + r % 4) * GP + pp * SB + 32 * q + col];
            dk[pp][q] = __builtin_amdgcn_mfma_f32_32x32x2f32(gt, u[r], dk[pp][q], 0, 0, 0);
          }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 8 * (r / 4) + 4 * hw + r % 4;
        const float ud = col_sum<HALF>(u[r] * du[r], col);
        const float dz = nz[r] > 1e-12f ? (du[r] - u[r] * ud) * inz[r] : du[r] * 1e12f;
        if (live_col && row < left) {
          const int at = row * dzs + p * HALF + col;
          if (a.out_bf16) dzb[at] = from_f32<bf16_t>(dz);
          else dzt[at] = dz;
          acc_ab[p] += dz;
        }
      }
    }
    wave_lds_fence();
  }
  // an address element that is not finite has left NaN in its column of every sub-key's sum
  bool odd = __ballot(!fin) != 0ull;
#pragma unroll
  for (int p = 0; p < NT; ++p) {
    bool bad = true;
#pragma unroll
    for (int q = 0; q < NSB; ++q)
#pragma unroll
      for (int r = 0; r < 16; ++r) bad = bad && !finite_f32(dk[p][q][r]);
    const unsigned long long b = __ballot(bad);
    odd = odd || (static_cast<uint32_t>(b) & static_cast<uint32_t>(b >> 32)) != 0u;   // a column's rows: both half-waves
  }
  if (lane == 0) s_odd[w] = odd;
  // block sums in a fixed order: waves -> LDS -> threads
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    acc_gb += __shfl_xor(acc_gb, off);
    acc_lam += __shfl_xor(acc_lam, off);
    acc_tau += __shfl_xor(acc_tau, off);
  }
#pragma unroll
  for (int p = 0; p < NT; ++p) acc_ab[p] += __shfl_xor(acc_ab[p], 32);
  __syncthreads();   // every wave's G is done with
  if (s_odd[0] | s_odd[1] | s_odd[2] | s_odd[3]) {   // rare
    __threadfence();   // the block's row gradients, written again by other threads
    __syncthreads();
    addr_grad_block<HALF, KP, InT>(a, albuf);
    return;
  }
  float* dkb = reinterpret_cast<float*>(albuf);
  unsigned char* tail = albuf + (addr_tile_lds(n_sub, HALF, NSB) -
                                 kAddrTileWaves * (sizeof(double) + sizeof(float) * (2 * HALF + 2)));
  double* redd = reinterpret_cast<double*>(tail);
  float* red = reinterpret_cast<float*>(tail + kAddrTileWaves * sizeof(double));
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int c = NT == 2 ? col : col - p * HALF;
    if (c < 0 || c >= HALF) continue;
#pragma unroll
    for (int q = 0; q < NSB; ++q)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = 32 * q + 8 * (r / 4) + 4 * hw + r % 4;
        if (i < n_sub) dkb[w * KS + (p * n_sub + i) * HALF + c] = dk[p][q][r];
      }
  }
  if (hw == 0) {
#pragma unroll
    for (int p = 0; p < NT; ++p)
      if (NT == 2 ? col < HALF : col < DA) red[w * (DA + 2) + p * HALF + col] = acc_ab[p];
  }
  if (lane == 0) {
    red[w * (DA + 2) + DA] = static_cast<float>(acc_tau);
    red[w * (DA + 2) + DA + 1] = static_cast<float>(acc_gb);
    redd[w] = acc_lam;
  }
  __syncthreads();
  const int64_t pid = (static_cast<int64_t>(blockIdx.x) * gridDim.z + blockIdx.z) * a.H + h;
  for (int c = tid; c < DA + 2; c += blockDim.x) {
    float s = 0.f;
    for (int q = 0; q < kAddrTileWaves; ++q) s += red[q * (DA + 2) + c];
    // record order: dtau, d gate bias, d addr_b[DA]
    const int f = c == DA ? 0 : c == DA + 1 ? 1 : 2 + c;
    a.part_f[pid * (2 + DA) + f] = s;
  }
  if (tid == 0) {
    double s = 0.0;
    for (int q = 0; q < kAddrTileWaves; ++q) s += redd[q];
    a.part_d[pid] = s;
  }
  for (int i = tid; i < KS; i += blockDim.x) {
    float s = 0.f;
    for (int q = 0; q < kAddrTileWaves; ++q) s += dkb[q * KS + i];
    a.part_k[pid * KS + i] = s;
  }
}

// The parameter gradients from the blocks' partial records, all in one launch (seven of them, each a few microseconds
// of launch and round trips, took 34 us of a backward of B=8, T=2048; this one takes 10): block ranges by what they sum, 64 items a
// block (reduce_item), in float64.
//   keys    whole sub-key rows, 64 / half a block; from the summed unit sub-key gradient dk^ the raw one (F.normalize
//           backward): dK = (dk^ - k^ <k^, dk^>) / |K|   (dk^ / 1e-12 below the floor)
//   fields  [H][2 + d_a]: dtau (times tau: the gradient with respect to log tau), the gate bias, addr_b
//   fades   [H]: lam dL/dlam
//   onorm   [H][dh]
struct GradSumsArgs {
  const float* pk;        // [n_rec][H][2][n_sub][half]
  const float* pf;        // [n_rec][H][2 + DA]
  const double* pd;       // [n_rec][H]
  const float* p1;        // [n_rb][H * dh]
  int n_rec, n_rb, H, DA, n_sub, half, n_onorm;
  int key_blocks, field_blocks, fade_blocks;   // the onorm blocks follow
  const float* keys[2];
  const float* log_scale;
  float* d_keys[2];
  float* d_log_scale;
  float* d_gate_bias;
  float* d_addr_b;
  float* d_log_decay;
  float* d_onorm;
};

__global__ void __launch_bounds__(64 * kRedGroups) grad_sums_kernel(GradSumsArgs a) {
  __shared__ double red[kRedGroups][64];
  __shared__ float dkn[64], key[64];
  const int l = threadIdx.x & 63;
  const bool first = threadIdx.x < 64;   // the lanes that hold the sums
  int blk = blockIdx.x;
  if (blk < a.key_blocks) {
    const int rows = 64 / a.half;
    const int row = blk * rows + l / a.half;   // [H][2][n_sub]
    const int n_rows = a.H * 2 * a.n_sub;
    const bool live = l / a.half < rows && row < n_rows;
    const int64_t i = static_cast<int64_t>(blk) * rows * a.half + l;
    const double s = reduce_item(a.pk, a.n_rec, static_cast<int64_t>(n_rows) * a.half, i, live, red);
    const int h = row / (2 * a.n_sub), part = (row / a.n_sub) & 1, sub = row % a.n_sub;
    const int64_t at = (static_cast<int64_t>(h) * a.n_sub + sub) * a.half + l % a.half;
    if (first) {
      dkn[l] = static_cast<float>(s);
      key[l] = live ? a.keys[part][at] : 0.f;
    }
    __syncthreads();
    if (!first || !live) return;
    const int c0 = l / a.half * a.half;
    float kk = 0.f;
    for (int c = 0; c < a.half; ++c) kk = fmaf(key[c0 + c], key[c0 + c], kk);
    const float nk = sqrtf(kk), inv = fmaxf(nk, 1e-12f);
    float dot = 0.f;
    for (int c = 0; c < a.half; ++c) dot = fmaf(key[c0 + c] / inv, dkn[c0 + c], dot);
    a.d_keys[part][at] = nk > 1e-12f ? (dkn[l] - key[l] / inv * dot) / nk : dkn[l] * 1e12f;
    return;
  }
  blk -= a.key_blocks;
  if (blk < a.field_blocks) {
    const int F = 2 + a.DA;
    const int64_t i = static_cast<int64_t>(blk) * 64 + l, n = static_cast<int64_t>(a.H) * F;
    const double s = reduce_item(a.pf, a.n_rec, n, i, i < n, red);
    if (!first || i >= n) return;
    const int h = static_cast<int>(i / F), f = static_cast<int>(i % F);
    if (f == 0) {
      if (a.d_log_scale) a.d_log_scale[h] = static_cast<float>(s * static_cast<double>(expf(a.log_scale[h])));
    } else if (f == 1) {
      if (a.d_gate_bias) a.d_gate_bias[h] = static_cast<float>(s);
    } else if (a.d_addr_b) {
      a.d_addr_b[h * a.DA + (f - 2)] = static_cast<float>(s);
    }
    return;
  }
  blk -= a.field_blocks;
  const bool fade = blk < a.fade_blocks;
  if (!fade) blk -= a.fade_blocks;
  const int64_t i = static_cast<int64_t>(blk) * 64 + l, n = fade ? a.H : a.n_onorm;
  const double s = fade ? reduce_item(a.pd, a.n_rec, n, i, i < n, red) : reduce_item(a.p1, a.n_rb, n, i, i < n, red);
  if (first && i < n) (fade ? a.d_log_decay : a.d_onorm)[i] = static_cast<float>(s);
}

// ---------------------------------------------------------------------------------------------------------------
// table read backward (TrainedSdm's embedding_bag, track4_onesdm_models.py:448-455)
//   dw[n][h][j]          = <values[h][slot_j], dy[n][h]>    (table_grad_kernel: the per-pick gradient the softmax
//                                                           backward takes; one wave per (token, head), lane l takes
//                                                           columns 4l, 4l + 256, ...)
//   d_values[h][s]       = sum over the picks (n, j) of slot s of w_j dy[n][h]   (table_values_grad_kernel: the picks
//                          sorted by (head, slot) with a stable radix sort and summed in pieces in pick order -- no
//                          float atomics, a fixed order)
// Four consecutive values of a row as they lie in memory: one load each, converted where they are used.  VEC: the rows
// start on a multiple of four values (checked on the host).  load_vals checks each address instead, and a load behind a
// branch of its own is waited for there, so a batch's loads run one after another (B=4, T=1024, rows of 768, k=16: values
// gradient 49 -> 42 us, per-pick gradients 23.5 -> 19.6 us).
template <typename T, bool VEC>
struct Quad {
  using Raw = typename std::conditional<sizeof(T) == 2, uint2, float4>::type;
  Raw r;
  __device__ __forceinline__ void load(const T* p) {
    if constexpr (VEC) {
      r = *reinterpret_cast<const Raw*>(p);
    } else {
      T* d = reinterpret_cast<T*>(&r);
#pragma unroll
      for (int k = 0; k < 4; ++k) d[k] = p[k];
    }
  }
  __device__ __forceinline__ void get(float (&v)[4]) const {
    if constexpr (sizeof(T) == 2) {
      v[0] = __uint_as_float(r.x << 16);
      v[1] = __uint_as_float(r.x & 0xffff0000u);
      v[2] = __uint_as_float(r.y << 16);
      v[3] = __uint_as_float(r.y & 0xffff0000u);
    } else {
      v[0] = r.x;
      v[1] = r.y;
      v[2] = r.z;
      v[3] = r.w;
    }
  }
};

inline bool quad_rows(const void* p, int64_t stride, sdm_rt_dtype t) {
  return reinterpret_cast<uintptr_t>(p) % (t == SDM_RT_BF16 ? 8 : 16) == 0 && stride % 4 == 0;
}

template <int KP, typename VT, typename DyT, bool VEC>
__global__ void __launch_bounds__(256) table_grad_kernel(const int32_t* __restrict__ slots,
                                                         const float* __restrict__ wts,
                                                         const VT* __restrict__ values, const DyT* __restrict__ dy,
                                                         int64_t dy_stride, float* __restrict__ dw, int B, int T,
                                                         int H, int M, int dh, int kk) {
  const int64_t wave = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (wave >= static_cast<int64_t>(B) * T * H) return;   // whole waves
  const int64_t n = wave / H;
  const int h = static_cast<int>(wave - n * H);
  const int b = static_cast<int>(n / T);
  const int t = static_cast<int>(n - static_cast<int64_t>(b) * T);
  const int64_t pb = ((static_cast<int64_t>(b) * H + h) * T + t) * KP;
  int sl[KP];
  float d[KP];
#pragma unroll
  for (int j = 0; j < KP; ++j) {
    sl[j] = min(max(slots[pb + j], 0), M - 1);   // pads (-1) and stray ids stay inside the table
    d[j] = 0.f;
  }
  (void)wts;
  const VT* tab = values + static_cast<int64_t>(h) * M * dh;
  for (int c0 = 4 * lane; c0 < dh; c0 += 256) {
    Quad<DyT, VEC> gq;
    gq.load(dy + n * dy_stride + static_cast<int64_t>(h) * dh + c0);
    // every pick's row, pads included (their dots are dropped below): unconditional loads issue together
    Quad<VT, VEC> vq[KP];
#pragma unroll
    for (int j = 0; j < KP; ++j) vq[j].load(tab + static_cast<int64_t>(sl[j]) * dh + c0);
    float g[4];
    gq.get(g);
#pragma unroll
    for (int j = 0; j < KP; ++j) {
      float v[4];
      vq[j].get(v);
#pragma unroll
      for (int e = 0; e < 4; ++e) d[j] = fmaf(g[e], v[e], d[j]);
    }
  }
#pragma unroll
  for (int j = 0; j < KP; ++j) {
    const float s = wave_sum(d[j]);
    if (lane == 0) dw[pb + j] = j < kk ? s : 0.f;
  }
}

__global__ void __launch_bounds__(256) zero_i32_kernel(int32_t* __restrict__ p, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0;
}

// sort keys of the picks: entry e of the [B][H][T][KP] pick arrays gets key h * M + slot (pads: H * M, after every
// real key) and value e; count[key] counts the live picks of each (head, slot)
__global__ void __launch_bounds__(256) pick_keys_kernel(const int32_t* __restrict__ slots, int64_t n_entries, int T,
                                                        int H, int KP, int M, int kk, int32_t* __restrict__ keys,
                                                        int32_t* __restrict__ vals, int32_t* __restrict__ count) {
  const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (e >= n_entries) return;
  const int j = static_cast<int>(e % KP);
  const int h = static_cast<int>((e / KP / T) % H);
  int key = H * M;
  if (j < kk) {
    const int s = min(max(slots[e], 0), M - 1);
    key = h * M + s;
    atomicAdd(&count[key], 1);   // integer counts: exact in any order
  }
  keys[e] = key;
  vals[e] = static_cast<int32_t>(e);
}

// d_values[h][s] = sum of w_e dy[n_e][h] over the picks e of (h, s), in two launches.  The sorted picks are cut every
// kValuesSeg entries and a wave sums one piece's runs of equal keys in pick order, lane l columns 4l, 4l + 256, ...: a
// run that is its whole row goes to d_values, one that crosses an edge of the piece to part: [2 s] continues a row
// begun before piece s, [2 s + 1] begins a row that goes on after it.  table_values_join_kernel adds a row's pieces in
// order and clears the rows without a pick.  The load follows the picks and not the rows: text repeats its tokens, so a
// few rows hold hundreds of picks, and with one wave per row the longest row's chain of batches was the kernel's time
// (B=4, T=1024, 4,096 rows of 768, k=16, a Zipf stream: 190 us; now 42 us and 10 for the join; the
// floor is the 101 MB of dy rows gathered through the caches).  Pieces of 32: the partial sums then take at most a
// quarter of the gathered bytes again, and 2,048 waves are all resident at three to a SIMD.
constexpr int kValuesSeg = 32;

template <typename DyT, bool VEC>
__global__ void __launch_bounds__(256) table_values_grad_kernel(const int32_t* __restrict__ sorted_keys,
                                                                const int32_t* __restrict__ sorted_vals,
                                                                const int32_t* __restrict__ offsets,
                                                                const float* __restrict__ wts,
                                                                const DyT* __restrict__ dy, int64_t dy_stride,
                                                                float* __restrict__ d_values,
                                                                float* __restrict__ part, int T, int H, int KP, int M,
                                                                int dh) {
  const int lane = threadIdx.x & 63;
  const int seg = __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x) * 4 + (threadIdx.x >> 6));
  const int live = offsets[H * M];   // the pads' key comes last
  const int64_t begin = static_cast<int64_t>(seg) * kValuesSeg;
  if (begin >= live) return;   // whole waves
  const int i_begin = static_cast<int>(begin);
  const int n = min(kValuesSeg, live - i_begin);
  const int before = i_begin > 0 ? sorted_keys[i_begin - 1] : -1;
  const int after = i_begin + n < live ? sorted_keys[i_begin + n] : -1;
  // up to CS column steps of 256 held in registers; the picks QS at a time: their indexes and weights, then every
  // row segment, all loads of a batch in flight together
  constexpr int CS = 4, QS = 8;
  for (int cb = 0; cb < dh; cb += 256 * CS) {
    float acc[CS][4];
#pragma unroll
    for (int s = 0; s < CS; ++s)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[s][c] = 0.f;
    int cur = sorted_keys[i_begin];
    bool first = true;   // the run of cur begins at the piece's first entry
    auto flush = [&](bool last) {
      float* dst = d_values + static_cast<int64_t>(cur) * dh;
      if (first && cur == before) {
        dst = part + 2 * static_cast<int64_t>(seg) * dh;
      } else if (last && cur == after) {
        dst = part + (2 * static_cast<int64_t>(seg) + 1) * dh;
      }
#pragma unroll
      for (int s = 0; s < CS; ++s) {
        const int c0 = cb + 256 * s + 4 * lane;
        if (c0 < dh) store_vals<4, float>(dst + c0, acc[s]);
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[s][c] = 0.f;
      }
    };
    for (int i0 = 0; i0 < n; i0 += QS) {
      int64_t ro[QS];
      float w[QS];
      int key[QS];
#pragma unroll
      for (int q = 0; q < QS; ++q) {
        const int i = i_begin + min(i0 + q, n - 1);
        const uint32_t e = static_cast<uint32_t>(sorted_vals[i]);   // ((b * H + h) * T + t) * KP + j, below 2^31
        const uint32_t u = e / static_cast<uint32_t>(KP);
        const uint32_t bh = u / static_cast<uint32_t>(T);
        const uint32_t b = bh / static_cast<uint32_t>(H);
        const uint32_t t = u - bh * static_cast<uint32_t>(T), h = bh - b * static_cast<uint32_t>(H);
        w[q] = i0 + q < n ? wts[e] : 0.f;
        key[q] = sorted_keys[i];
        ro[q] = (static_cast<int64_t>(b) * T + t) * dy_stride + static_cast<int64_t>(h) * dh;
      }
      Quad<DyT, VEC> gq[QS][CS];
#pragma unroll
      for (int q = 0; q < QS; ++q) {
#pragma unroll
        for (int s = 0; s < CS; ++s) {
          const int c0 = cb + 256 * s + 4 * lane;
          if (c0 < dh) gq[q][s].load(dy + ro[q] + c0);
        }
      }
#pragma unroll
      for (int q = 0; q < QS; ++q) {
        if (key[q] != cur) {   // the same for the whole wave
          flush(false);
          cur = key[q];
          first = false;
        }
        if (i0 + q < n) {   // past the piece's end nothing is added: 0 * dy would keep an infinity's NaN
#pragma unroll
          for (int s = 0; s < CS; ++s) {
            float g[4];
            gq[q][s].get(g);
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[s][c] = fmaf(w[q], g[c], acc[s][c]);
          }
        }
      }
    }
    flush(true);
  }
}

// d_values rows without a pick: zero; rows cut over several pieces: their partial sums in order; one wave per row
__global__ void __launch_bounds__(256) table_values_join_kernel(const int32_t* __restrict__ offsets,
                                                                const int32_t* __restrict__ count,
                                                                const float* __restrict__ part,
                                                                float* __restrict__ d_values, int n_rows, int dh) {
  const int row = __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x) * 4 + (threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;
  if (row >= n_rows) return;   // whole waves
  const int off = offsets[row], cnt = count[row];
  const int s0 = off / kValuesSeg, s1 = (off + max(cnt, 1) - 1) / kValuesSeg;
  if (cnt > 0 && s0 == s1) return;   // written by its one piece
  for (int c0 = 4 * lane; c0 < dh; c0 += 256) {
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    if (cnt > 0) {
      load_vals<4, float>(part + (2 * static_cast<int64_t>(s0) + 1) * dh + c0, acc);
#pragma unroll 8
      for (int s = s0 + 1; s <= s1; ++s) {
        float v[4];
        load_vals<4, float>(part + 2 * static_cast<int64_t>(s) * dh + c0, v);
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] += v[c];
      }
    }
    store_vals<4, float>(d_values + static_cast<int64_t>(row) * dh + c0, acc);
  }
}

// ---------------------------------------------------------------------------------------------------------------
// host side of the backward
// waves per addr_grad block: as many as LDS holds, up to addr_grad_max_waves
int addr_grad_waves(int n_sub, int half, int KP) {
  for (int w = addr_grad_max_waves(KP); w >= 1; --w)
    if (addr_grad_lds(n_sub, half, w) <= kLdsBytes) return w;
  return 0;
}

// 32-token tiles per wave of addr_grad_tile_kernel: the fewest that leave no more than two blocks for each of the 256
// compute units, at most 8; 0 for more than 64 sub-keys per half, which addr_grad_kernel serves.  Two blocks fit a
// compute unit by their registers, and by their LDS with up to 32 sub-keys (43 KB a block); with more (84 KB) one fits,
// and the second of a unit's two follows the first
int addr_tiles(const Plan& p, int sets) {
  if (p.n_sub > 64) return 0;
  const int64_t N = static_cast<int64_t>(p.B) * p.T;
  int tiles = 1;
  while (tiles < 8 && (N + 128 * tiles - 1) / (128 * tiles) * p.H * sets > 512) ++tiles;
  return tiles;
}

// tokens per block of the addressing backward
int64_t addr_block_tokens(int tiles, int waves) {
  return tiles ? static_cast<int64_t>(tiles) * kAddrTile * kAddrTileWaves
               : static_cast<int64_t>(waves) * kAddrGradWaveTokens;
}

struct GradPlan {
  Plan p;
  int cw, n_cg, n_xg, n_rb, n_blk, addr_waves, tiles;   // n_xg: column groups of chunk_grad_kernel
  size_t off_dnum, off_dden, off_dv, off_dotw, off_dotr, off_p1, off_pf, off_pd, off_pk, off_chains, total;
};

// widest column group (32, 16, 8) whose grad_scan slab fits in LDS
int grad_columns(const Plan& p) {
  for (int cw : {32, 16, 8})
    if (p.dh % cw == 0 && GradScanLds(p.M, p.pitch, cw).total <= kLdsBytes) return cw;
  return 0;
}

int make_grad_plan(const sdm_rt_dims* d, GradPlan* g) {
  int rc = make_plan(d, &g->p);
  if (rc) return rc;
  const Plan& p = g->p;
  if (p.d_a > 64) return set_err(SDM_RT_EUNSUPPORTED, "backward: addr_dim %d exceeds 64", p.d_a);
  g->cw = grad_columns(p);
  if (!g->cw) return set_err(SDM_RT_EUNSUPPORTED, "backward: M = %d locations do not fit a slab in LDS", p.M);
  g->addr_waves = addr_grad_waves(p.n_sub, p.half, p.pitch);
  if (!g->addr_waves) return set_err(SDM_RT_EUNSUPPORTED, "backward: n_sub = %d sub-keys do not fit in LDS", p.n_sub);
  g->n_cg = p.dh / g->cw;
  g->n_xg = (p.dh + 63) / 64;
  const int64_t N = static_cast<int64_t>(p.B) * p.T;
  g->n_rb = static_cast<int>((N + kReadGradRows - 1) / kReadGradRows);
  g->tiles = addr_tiles(p, 2);
  const int64_t tpb = addr_block_tokens(g->tiles, g->addr_waves);
  g->n_blk = static_cast<int>((N + tpb - 1) / tpb);
  const size_t hd = static_cast<size_t>(p.H) * p.dh;
  const size_t picks = static_cast<size_t>(N) * p.H * p.pitch;
  size_t o = 0;
  g->off_dnum = o;
  o = align_up(o + sizeof(float) * N * hd, 256);
  g->off_dden = o;
  o = align_up(o + sizeof(float) * N * p.H, 256);
  g->off_dv = o;
  o = align_up(o + sizeof(float) * N * hd, 256);
  g->off_dotw = o;   // the scans' column groups, then chunk_grad_kernel's
  o = align_up(o + sizeof(float) * (g->n_cg + g->n_xg) * picks, 256);
  g->off_dotr = o;
  o = align_up(o + sizeof(float) * (g->n_cg + g->n_xg) * picks, 256);
  g->off_p1 = o;
  o = align_up(o + sizeof(float) * g->n_rb * hd, 256);
  g->off_pf = o;
  o = align_up(o + sizeof(float) * 2 * g->n_blk * p.H * (2 + p.d_a), 256);
  g->off_pd = o;
  o = align_up(o + sizeof(double) * 2 * g->n_blk * p.H, 256);
  g->off_pk = o;
  o = align_up(o + sizeof(float) * 2 * g->n_blk * p.H * 2 * static_cast<size_t>(p.n_sub) * p.half, 256);
  g->off_chains = o;   // the chain plans of one scan direction at a time
  o = align_up(o + static_cast<size_t>(p.B) * p.H * p.n_chunks * chain_stride(p.pitch), 256);
  g->total = o;
  return SDM_RT_OK;
}

template <int CW, int KP, bool REV, typename WT, typename RT>
int launch_grad_scan_t(const GradPlan& g, const GradScanArgs& a, const ChainArgs& c, hipStream_t st) {
  {
    hipLaunchKernelGGL((chain_plan_kernel<KP, REV>), dim3(a.n_chunks, a.H, a.B), dim3(64),
                       sizeof(unsigned long long) * a.M, st, c);
    if (int rc = check_launch("chain plan")) return rc;
  }
  const size_t lds = GradScanLds(g.p.M, KP, CW).total;
  static const hipError_t attr =
      hipFuncSetAttribute(reinterpret_cast<const void*>(&grad_scan_kernel<CW, KP, REV, WT, RT>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kLdsBytes));
  if (attr != hipSuccess) return set_err(SDM_RT_ELAUNCH, "grad scan: cannot enable %zu bytes of LDS", kLdsBytes);
  dim3 grid(g.n_cg, g.p.H, g.p.B);
  hipLaunchKernelGGL((grad_scan_kernel<CW, KP, REV, WT, RT>), grid, dim3(kGradScanThreads), lds, st, a);
  return check_launch("grad scan");
}

template <bool REV, typename WT, typename RT>
int launch_grad_scan(const GradPlan& g, const GradScanArgs& a, const ChainArgs& ch, hipStream_t st) {
  const bool k8 = g.p.pitch == 8;
  switch (g.cw) {
    case 32: return k8 ? launch_grad_scan_t<32, 8, REV, WT, RT>(g, a, ch, st) : launch_grad_scan_t<32, 16, REV, WT, RT>(g, a, ch, st);
    case 16: return k8 ? launch_grad_scan_t<16, 8, REV, WT, RT>(g, a, ch, st) : launch_grad_scan_t<16, 16, REV, WT, RT>(g, a, ch, st);
    default: return k8 ? launch_grad_scan_t<8, 8, REV, WT, RT>(g, a, ch, st) : launch_grad_scan_t<8, 16, REV, WT, RT>(g, a, ch, st);
  }
}

// the parameter gradients asked for (null outputs are left out)
int launch_grad_sums(GradSumsArgs a, hipStream_t st) {
  const int rows = 64 / a.half;
  a.key_blocks = a.d_keys[0] ? (a.H * 2 * a.n_sub + rows - 1) / rows : 0;
  a.field_blocks = (a.H * (2 + a.DA) + 63) / 64;
  a.fade_blocks = a.d_log_decay ? (a.H + 63) / 64 : 0;
  const int blocks = a.key_blocks + a.field_blocks + a.fade_blocks + (a.d_onorm ? (a.n_onorm + 63) / 64 : 0);
  hipLaunchKernelGGL(grad_sums_kernel, dim3(blocks), dim3(64 * kRedGroups), 0, st, a);
  return check_launch("gradient sums");
}

template <typename VT>
int launch_chunk_grad(const GradPlan& g, const ChunkGradArgs& a, hipStream_t st) {
  const Plan& p = g.p;
  const dim3 grid(p.n_chunks, p.H * g.n_xg, p.B);
  const size_t lds = ChunkGradLds(p.M, p.pitch).total;
  if (p.pitch == 8) {
    static const bool ok = allow_lds(reinterpret_cast<const void*>(&chunk_grad_kernel<8, VT>));
    if (!ok) return lds_err("chunk grad");
    hipLaunchKernelGGL((chunk_grad_kernel<8, VT>), grid, dim3(kGradScanThreads), lds, st, a);
  } else {
    static const bool ok = allow_lds(reinterpret_cast<const void*>(&chunk_grad_kernel<16, VT>));
    if (!ok) return lds_err("chunk grad");
    hipLaunchKernelGGL((chunk_grad_kernel<16, VT>), grid, dim3(kGradScanThreads), lds, st, a);
  }
  return check_launch("chunk grad");
}

template <int HALF, typename InT>
struct AddrGradLaunch {
  template <int NSB, int KP>
  static int run_tiles(const GradPlan& g, AddrGradArgs a, hipStream_t st) {
    static const bool ok = allow_lds(reinterpret_cast<const void*>(&addr_grad_tile_kernel<HALF, NSB, KP, InT>));
    if (!ok) return lds_err("addr grad");
    a.wave_tokens = g.tiles * kAddrTile;
    hipLaunchKernelGGL((addr_grad_tile_kernel<HALF, NSB, KP, InT>), dim3(g.n_blk, g.p.H, 2 - a.set0),
                       dim3(64 * kAddrTileWaves), addr_tile_lds(g.p.n_sub, HALF, NSB), st, a);
    return check_launch("addr grad");
  }

  static int run(const GradPlan& g, AddrGradArgs a, hipStream_t st) {
    const Plan& p = g.p;
    // the tile kernel's offsets inside a tile are 32 bits
    const int64_t far = std::max(std::max(a.kz_stride, a.qz_stride), std::max(a.dz_stride[0], a.dz_stride[1]));
    if (g.tiles && far < (1 << 25)) {
      if (p.n_sub <= 32) return p.pitch == 8 ? run_tiles<1, 8>(g, a, st) : run_tiles<1, 16>(g, a, st);
      return p.pitch == 8 ? run_tiles<2, 8>(g, a, st) : run_tiles<2, 16>(g, a, st);
    }
    a.wave_tokens = static_cast<int>((addr_block_tokens(g.tiles, g.addr_waves) + g.addr_waves - 1) / g.addr_waves);
    const size_t lds = addr_grad_lds(p.n_sub, HALF, g.addr_waves);
    dim3 grid(g.n_blk, p.H, 2 - a.set0);
    dim3 block(64 * g.addr_waves);
    if (p.pitch == 8) {
      static const bool ok = allow_lds(reinterpret_cast<const void*>(&addr_grad_kernel<HALF, 8, InT>));
      if (!ok) return lds_err("addr grad");
      hipLaunchKernelGGL((addr_grad_kernel<HALF, 8, InT>), grid, block, lds, st, a);
    } else {
      static const bool ok = allow_lds(reinterpret_cast<const void*>(&addr_grad_kernel<HALF, 16, InT>));
      if (!ok) return lds_err("addr grad");
      hipLaunchKernelGGL((addr_grad_kernel<HALF, 16, InT>), grid, block, lds, st, a);
    }
    return check_launch("addr grad");
  }
};

int check_saved(const sdm_rt_saved* s, bool need_den) {
  if (!s) return set_err(SDM_RT_EINVAL, "saved is NULL");
  if (!s->slots_w || !s->weights_w || !s->scores_w || !s->slots_r || !s->weights_r || !s->scores_r || !s->read)
    return set_err(SDM_RT_EINVAL, "saved: picks, weights, scores and read must not be NULL");
  if (need_den && !s->den) return set_err(SDM_RT_EINVAL, "saved: den must not be NULL for the mean read");
  return SDM_RT_OK;
}

// workspace of sdm_rt_table_backward: per-pick gradients, addressing partials (read set only), float64 sums
struct TablePlan {
  Plan p;
  int n_blk, addr_waves, tiles, key_bits;
  int64_t n_entries;
  size_t off_dw, off_pf, off_pd, off_pk, off_keys, off_count, off_offsets, off_part, off_cub, cub_bytes, total;
};

// pieces of the sorted picks in the value-table gradient
int64_t values_pieces(int64_t n_entries) { return (n_entries + kValuesSeg - 1) / kValuesSeg; }

int make_table_plan(const sdm_rt_dims* d, TablePlan* g) {
  int rc = make_plan(d, &g->p, false);
  if (rc) return rc;
  const Plan& p = g->p;
  if (p.d_a > 64) return set_err(SDM_RT_EUNSUPPORTED, "table backward: addr_dim %d exceeds 64", p.d_a);
  if (p.dh < 4 || p.dh % 4 != 0) return set_err(SDM_RT_EUNSUPPORTED, "head_dim %d must be a positive multiple of 4", p.dh);
  g->addr_waves = addr_grad_waves(p.n_sub, p.half, p.pitch);
  if (!g->addr_waves) return set_err(SDM_RT_EUNSUPPORTED, "table backward: n_sub = %d sub-keys do not fit in LDS", p.n_sub);
  const int64_t N = static_cast<int64_t>(p.B) * p.T;
  g->tiles = addr_tiles(p, 1);
  const int64_t tpb = addr_block_tokens(g->tiles, g->addr_waves);
  g->n_blk = static_cast<int>((N + tpb - 1) / tpb);
  const size_t KSH = static_cast<size_t>(p.H) * 2 * p.n_sub * p.half;
  size_t o = 0;
  g->off_dw = o;
  o = align_up(o + sizeof(float) * N * p.H * p.pitch, 256);
  g->off_pf = o;
  o = align_up(o + sizeof(float) * g->n_blk * p.H * (2 + p.d_a), 256);
  g->off_pd = o;
  o = align_up(o + sizeof(double) * g->n_blk * p.H, 256);
  g->off_pk = o;
  o = align_up(o + sizeof(float) * g->n_blk * KSH, 256);
  // the value-table gradient: sort keys and values (in and out), per-row counts and offsets, hipCUB's scratch
  g->n_entries = N * p.H * p.pitch;
  if (g->n_entries > 0x7fffffffLL) return set_err(SDM_RT_EUNSUPPORTED, "table backward: too many picks");
  const int n_keys = p.H * p.M + 1;
  g->key_bits = 1;
  while ((1LL << g->key_bits) <= n_keys) ++g->key_bits;
  g->off_keys = o;
  o = align_up(o + 4 * sizeof(int32_t) * static_cast<size_t>(g->n_entries), 256);
  g->off_count = o;
  o = align_up(o + sizeof(int32_t) * n_keys, 256);
  g->off_offsets = o;
  o = align_up(o + sizeof(int32_t) * n_keys, 256);
  g->off_part = o;
  o = align_up(o + 2 * sizeof(float) * static_cast<size_t>(values_pieces(g->n_entries)) * p.dh, 256);
  size_t sort_bytes = 0, scan_bytes = 0;
  if (hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, static_cast<const int32_t*>(nullptr),
                                         static_cast<int32_t*>(nullptr), static_cast<const int32_t*>(nullptr),
                                         static_cast<int32_t*>(nullptr), static_cast<int>(g->n_entries), 0,
                                         g->key_bits) != hipSuccess ||
      hipcub::DeviceScan::ExclusiveSum(nullptr, scan_bytes, static_cast<const int32_t*>(nullptr),
                                       static_cast<int32_t*>(nullptr), n_keys) != hipSuccess)
    return set_err(SDM_RT_ELAUNCH, "table backward: sort scratch size query failed");
  g->cub_bytes = sort_bytes > scan_bytes ? sort_bytes : scan_bytes;
  g->off_cub = o;
  o = align_up(o + g->cub_bytes, 256);
  g->total = o;
  return SDM_RT_OK;
}

}  // namespace sdmrt

using namespace sdmrt;

// ---------------------------------------------------------------------------------------------------------------
// C ABI of the backward
extern "C" {

int sdm_rt_forward_train(const sdm_rt_dims* dims, const sdm_rt_params* params, const void* kz,
                         int64_t kz_row_stride, const void* qz, int64_t qz_row_stride, const void* v,
                         int64_t v_row_stride, const void* gate_logits, int64_t gate_row_stride,
                         sdm_rt_dtype in_dtype, const uint8_t* reset, void* r_out, int64_t out_row_stride,
                         sdm_rt_dtype out_dtype, const sdm_rt_saved* saved, void* workspace, size_t workspace_bytes,
                         void* stream) {
  g_err[0] = 0;
  Plan p;
  int rc = make_plan(dims, &p);
  if (rc) return rc;
  if ((rc = check_params(params, dims->out_norm != 0))) return rc;
  if ((rc = check_dtype(in_dtype, "in_dtype"))) return rc;
  if ((rc = check_dtype(out_dtype, "out_dtype"))) return rc;
  if (p.B == 0 || p.T == 0) return SDM_RT_OK;
  if ((rc = check_saved(saved, dims->read_mean != 0))) return rc;
  if (!kz || !qz || !v || !r_out) return set_err(SDM_RT_EINVAL, "kz, qz, v and r_out must not be NULL");
  if (dims->write_gate && !gate_logits) return set_err(SDM_RT_EINVAL, "write_gate is set but gate_logits is NULL");
  const int64_t wa = static_cast<int64_t>(p.H) * p.d_a;
  const int64_t wv = static_cast<int64_t>(p.H) * p.dh;
  if (kz_row_stride < wa || qz_row_stride < wa) return set_err(SDM_RT_EINVAL, "kz/qz row stride < heads * addr_dim");
  if (v_row_stride < wv) return set_err(SDM_RT_EINVAL, "v_row_stride < heads * head_dim");
  if (gate_logits && gate_row_stride < p.H) return set_err(SDM_RT_EINVAL, "gate_row_stride < heads");
  if (out_row_stride < wv) return set_err(SDM_RT_EINVAL, "out_row_stride < heads * head_dim");
  if (!workspace || workspace_bytes < p.total)
    return set_err(SDM_RT_ENOSPACE, "workspace %zu bytes < required %zu", workspace_bytes, p.total);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const void* gl = dims->write_gate ? gate_logits : nullptr;

  CoreIO io{};
  io.kz = kz;
  io.kz_stride = kz_row_stride;
  io.qz = qz;
  io.qz_stride = qz_row_stride;
  io.v = v;
  io.v_stride = v_row_stride;
  io.gate_logits = gl;
  io.g_stride = gate_row_stride;
  io.in_dtype = in_dtype;
  io.reset = reset;
  io.r_out = r_out;
  io.r_stride = out_row_stride;
  io.out_dtype = out_dtype;
  io.saved = saved;   // the plan kernel's picks, weights (gate included) and scores
  io.read_out = saved->read;
  io.den_out = dims->read_mean ? saved->den : nullptr;
  return run_core(p, dims, params, io, workspace, workspace_bytes, st);
}

size_t sdm_rt_backward_workspace_bytes(const sdm_rt_dims* dims) {
  GradPlan g;
  if (make_grad_plan(dims, &g) != SDM_RT_OK) return 0;
  return g.total;
}

int sdm_rt_backward(const sdm_rt_dims* dims, const sdm_rt_params* params, const void* kz, int64_t kz_row_stride,
                    const void* qz, int64_t qz_row_stride, const void* v, int64_t v_row_stride,
                    const void* gate_logits, int64_t gate_row_stride, sdm_rt_dtype in_dtype, const uint8_t* reset,
                    const sdm_rt_saved* saved, const void* dy, int64_t dy_row_stride, sdm_rt_dtype dy_dtype,
                    const sdm_rt_grads* grads, void* workspace, size_t workspace_bytes, void* stream) {
  return sdm_rt_backward_typed(dims, params, kz, kz_row_stride, qz, qz_row_stride, v, v_row_stride, gate_logits,
                               gate_row_stride, in_dtype, reset, saved, dy, dy_row_stride, dy_dtype, grads, SDM_RT_F32,
                               workspace, workspace_bytes, stream);
}

int sdm_rt_backward_typed(const sdm_rt_dims* dims, const sdm_rt_params* params, const void* kz, int64_t kz_row_stride,
                          const void* qz, int64_t qz_row_stride, const void* v, int64_t v_row_stride,
                          const void* gate_logits, int64_t gate_row_stride, sdm_rt_dtype in_dtype,
                          const uint8_t* reset, const sdm_rt_saved* saved, const void* dy, int64_t dy_row_stride,
                          sdm_rt_dtype dy_dtype, const sdm_rt_grads* grads, sdm_rt_dtype grad_dtype, void* workspace,
                          size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  GradPlan g;
  int rc = make_grad_plan(dims, &g);
  if (rc) return rc;
  const Plan& p = g.p;
  if ((rc = check_params(params, dims->out_norm != 0))) return rc;
  if ((rc = check_dtype(in_dtype, "in_dtype"))) return rc;
  if ((rc = check_dtype(dy_dtype, "dy_dtype"))) return rc;
  if ((rc = check_dtype(grad_dtype, "grad_dtype"))) return rc;
  if (!grads) return set_err(SDM_RT_EINVAL, "grads is NULL");
  if (p.B == 0 || p.T == 0) return SDM_RT_OK;
  if ((rc = check_saved(saved, dims->read_mean != 0))) return rc;
  if (!kz || !qz || !v || !dy) return set_err(SDM_RT_EINVAL, "kz, qz, v and dy must not be NULL");
  if (dims->write_gate && !gate_logits) return set_err(SDM_RT_EINVAL, "write_gate is set but gate_logits is NULL");
  if (!grads->d_kz || !grads->d_qz || !grads->d_v)
    return set_err(SDM_RT_EINVAL, "grads: d_kz, d_qz and d_v must not be NULL");
  if (dims->write_gate && !grads->d_gate_logits)
    return set_err(SDM_RT_EINVAL, "grads: d_gate_logits must not be NULL when write_gate is set");
  const int64_t wa = static_cast<int64_t>(p.H) * p.d_a;
  const int64_t wv = static_cast<int64_t>(p.H) * p.dh;
  if (kz_row_stride < wa || qz_row_stride < wa) return set_err(SDM_RT_EINVAL, "kz/qz row stride < heads * addr_dim");
  if (v_row_stride < wv || dy_row_stride < wv) return set_err(SDM_RT_EINVAL, "v/dy row stride < heads * head_dim");
  if (gate_logits && gate_row_stride < p.H) return set_err(SDM_RT_EINVAL, "gate_row_stride < heads");
  if (grads->d_kz_row_stride < wa || grads->d_qz_row_stride < wa)
    return set_err(SDM_RT_EINVAL, "grads: d_kz/d_qz row stride < heads * addr_dim");
  if (grads->d_v_row_stride < wv) return set_err(SDM_RT_EINVAL, "grads: d_v row stride < heads * head_dim");
  if (dims->write_gate && grads->d_gate_row_stride < p.H)
    return set_err(SDM_RT_EINVAL, "grads: d_gate_logits row stride < heads");
  if (!workspace || workspace_bytes < g.total)
    return set_err(SDM_RT_ENOSPACE, "workspace %zu bytes < required %zu", workspace_bytes, g.total);
  hipStream_t st = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  float* dnum = reinterpret_cast<float*>(ws + g.off_dnum);
  float* dden = reinterpret_cast<float*>(ws + g.off_dden);
  float* dotw = reinterpret_cast<float*>(ws + g.off_dotw);
  float* dotr = reinterpret_cast<float*>(ws + g.off_dotr);
  float* p1 = reinterpret_cast<float*>(ws + g.off_p1);
  float* pf = reinterpret_cast<float*>(ws + g.off_pf);
  double* pd = reinterpret_cast<double*>(ws + g.off_pd);
  float* pk = reinterpret_cast<float*>(ws + g.off_pk);
  const int64_t N = static_cast<int64_t>(p.B) * p.T;
  const float* onw = dims->out_norm ? params->onorm_w : nullptr;

  // 1. read-out backward
  {
    dim3 grid(g.n_rb, p.H);
    if (dy_dtype == SDM_RT_BF16) {
      hipLaunchKernelGGL((p.dh <= 64 ? read_grad_kernel<bf16_t, 1> : read_grad_kernel<bf16_t, 8>), grid, dim3(256), 0, st, static_cast<const bf16_t*>(dy),
                         dy_row_stride, saved->read, saved->den, onw, dnum, dden, p1, N, p.H, p.dh, dims->read_mean,
                         dims->read_eps, dims->out_norm_eps);
    } else {
      hipLaunchKernelGGL((p.dh <= 64 ? read_grad_kernel<float, 1> : read_grad_kernel<float, 8>), grid, dim3(256), 0, st, static_cast<const float*>(dy),
                         dy_row_stride, saved->read, saved->den, onw, dnum, dden, p1, N, p.H, p.dh, dims->read_mean,
                         dims->read_eps, dims->out_norm_eps);
    }
    if ((rc = check_launch("read grad"))) return rc;
  }
  // 2. the chunks' own writes: parts of dwr, dww and dV
  float* dv_in = reinterpret_cast<float*>(ws + g.off_dv);
  {
    ChunkGradArgs a{};
    a.slot[0] = saved->slots_w;
    a.slot[1] = saved->slots_r;
    a.wt[0] = saved->weights_w;
    a.wt[1] = saved->weights_r;
    a.v = v;
    a.v_stride = v_row_stride;
    a.dnum = dnum;
    a.dden = dden;
    a.reset = reset;
    a.decay = params->decay;
    const int64_t picks = N * p.H * p.pitch;
    a.dot_w = dotw + g.n_cg * picks;
    a.dot_r = dotr + g.n_cg * picks;
    a.dv = dv_in;
    a.B = p.B;
    a.T = p.T;
    a.H = p.H;
    a.dh = p.dh;
    a.M = p.M;
    a.kk = p.kk;
    a.n_xg = g.n_xg;
    rc = in_dtype == SDM_RT_BF16 ? launch_chunk_grad<bf16_t>(g, a, st) : launch_chunk_grad<float>(g, a, st);
    if (rc) return rc;
  }
  // 3. the carried memory: forward replay (dwr), then the reverse scan (dww and dV)
  for (int rev = 0; rev < 2; ++rev) {
    ChainArgs c{};
    c.w_slot = rev ? saved->slots_r : saved->slots_w;
    c.w_wt = rev ? saved->weights_r : saved->weights_w;
    c.reset = reset;
    c.decay = params->decay;
    c.chains = reinterpret_cast<unsigned char*>(ws + g.off_chains);
    c.B = p.B;
    c.T = p.T;
    c.H = p.H;
    c.M = p.M;
    c.kk = p.kk;
    c.n_chunks = p.n_chunks;
    GradScanArgs a{};
    a.r_slot = rev ? saved->slots_w : saved->slots_r;
    a.r_wt = rev ? saved->weights_w : saved->weights_r;
    a.wv = rev ? dnum : v;
    a.wv_stride = rev ? wv : v_row_stride;
    a.wc = rev ? dden : nullptr;
    a.rv = rev ? v : dnum;
    a.rv_stride = rev ? v_row_stride : wv;
    a.rc = rev ? nullptr : dden;
    a.decay = params->decay;
    a.dot_out = rev ? dotw : dotr;
    if (rev) {
      a.sum_in = dv_in;
      a.sum_out = grads->d_v;
      a.sum_stride = grads->d_v_row_stride;
      a.sum_bf16 = grad_dtype == SDM_RT_BF16;
    }
    a.B = p.B;
    a.T = p.T;
    a.H = p.H;
    a.dh = p.dh;
    a.M = p.M;
    a.kk = p.kk;
    a.n_chunks = p.n_chunks;
    a.chains = c.chains;
    auto aligned = [](const void* p, int64_t stride, size_t piece) {   // every row's pieces start on their size
      return reinterpret_cast<uintptr_t>(p) % piece == 0 && stride % static_cast<int64_t>(piece) == 0;
    };
    const size_t in_es = in_dtype == SDM_RT_BF16 ? 2 : 4, cpl = g.cw / 8;
    a.vec = aligned(a.r_slot, 0, 16) && aligned(a.r_wt, 0, 16) &&
            aligned(v, v_row_stride * static_cast<int64_t>(in_es), in_es * cpl);
    const bool b16 = in_dtype == SDM_RT_BF16;
    rc = rev ? (b16 ? launch_grad_scan<true, float, bf16_t>(g, a, c, st) : launch_grad_scan<true, float, float>(g, a, c, st))
             : (b16 ? launch_grad_scan<false, bf16_t, float>(g, a, c, st)
                    : launch_grad_scan<false, float, float>(g, a, c, st));
    if (rc) return rc;
  }
  // 4. softmax, gate and address backward
  {
    AddrGradArgs a{};
    a.kz = kz;
    a.kz_stride = kz_row_stride;
    a.qz = qz;
    a.qz_stride = qz_row_stride;
    a.gl = dims->write_gate ? gate_logits : nullptr;
    a.g_stride = gate_row_stride;
    a.keys[0] = params->keys1;
    a.keys[1] = params->keys2;
    a.addr_b = params->addr_b;
    a.log_scale = params->log_scale;
    a.gate_bias = params->gate_bias;
    a.slot[0] = saved->slots_w;
    a.slot[1] = saved->slots_r;
    a.wt[0] = saved->weights_w;
    a.wt[1] = saved->weights_r;
    a.score[0] = saved->scores_w;
    a.score[1] = saved->scores_r;
    a.dot[0] = dotw;
    a.dot[1] = dotr;
    a.n_cg = g.n_cg + g.n_xg;
    a.dz[0] = grads->d_kz;
    a.dz[1] = grads->d_qz;
    a.dz_stride[0] = grads->d_kz_row_stride;
    a.dz_stride[1] = grads->d_qz_row_stride;
    a.dgl = dims->write_gate ? grads->d_gate_logits : nullptr;
    a.dgl_stride = grads->d_gate_row_stride;
    a.out_bf16 = grad_dtype == SDM_RT_BF16;
    a.part_f = pf;
    a.part_d = pd;
    a.part_k = pk;
    a.B = p.B;
    a.T = p.T;
    a.H = p.H;
    a.n_sub = p.n_sub;
    a.kk = p.kk;
    rc = in_dtype == SDM_RT_BF16 ? by_half<AddrGradLaunch, bf16_t>(p.half, g, a, st)
                                 : by_half<AddrGradLaunch, float>(p.half, g, a, st);
    if (rc) return rc;
  }
  // 5. parameter sums
  {
    if ((grads->d_keys1 == nullptr) != (grads->d_keys2 == nullptr))
      return set_err(SDM_RT_EINVAL, "grads: give both d_keys1 and d_keys2");
    GradSumsArgs a{};
    a.pk = pk;
    a.pf = pf;
    a.pd = pd;
    a.p1 = p1;
    a.n_rec = 2 * g.n_blk;
    a.n_rb = g.n_rb;
    a.H = p.H;
    a.DA = p.d_a;
    a.n_sub = p.n_sub;
    a.half = p.half;
    a.n_onorm = static_cast<int>(wv);
    a.keys[0] = params->keys1;
    a.keys[1] = params->keys2;
    a.log_scale = params->log_scale;
    a.d_keys[0] = grads->d_keys1;
    a.d_keys[1] = grads->d_keys2;
    a.d_log_scale = grads->d_log_scale;
    a.d_gate_bias = grads->d_gate_bias;
    a.d_addr_b = grads->d_addr_b;
    a.d_log_decay = grads->d_log_decay;
    a.d_onorm = onw ? grads->d_onorm_w : nullptr;
    if ((rc = launch_grad_sums(a, st))) return rc;
  }
  return SDM_RT_OK;
}

size_t sdm_rt_table_backward_workspace_bytes(const sdm_rt_dims* dims) {
  TablePlan g;
  if (make_table_plan(dims, &g) != SDM_RT_OK) return 0;
  return g.total;
}

int sdm_rt_table_backward(const sdm_rt_dims* dims, const sdm_rt_params* params, const void* q, int64_t q_row_stride,
                          sdm_rt_dtype in_dtype, const int32_t* slots, const float* weights, const float* scores,
                          const void* values, sdm_rt_dtype values_dtype, const void* dy, int64_t dy_row_stride,
                          sdm_rt_dtype dy_dtype, float* d_q, int64_t d_q_row_stride, float* d_values,
                          float* d_keys1, float* d_keys2, float* d_log_scale, void* workspace,
                          size_t workspace_bytes, void* stream) {
  g_err[0] = 0;
  TablePlan g;
  int rc = make_table_plan(dims, &g);
  if (rc) return rc;
  const Plan& p = g.p;
  if ((rc = check_params(params, false, false))) return rc;
  if ((rc = check_dtype(in_dtype, "in_dtype"))) return rc;
  if ((rc = check_dtype(values_dtype, "values_dtype"))) return rc;
  if ((rc = check_dtype(dy_dtype, "dy_dtype"))) return rc;
  if (p.B == 0 || p.T == 0) return SDM_RT_OK;
  if (!q || !slots || !weights || !scores || !values || !dy || !d_q || !d_values)
    return set_err(SDM_RT_EINVAL, "q, slots, weights, scores, values, dy, d_q and d_values must not be NULL");
  if ((d_keys1 == nullptr) != (d_keys2 == nullptr)) return set_err(SDM_RT_EINVAL, "give both d_keys1 and d_keys2");
  const int64_t wa = static_cast<int64_t>(p.H) * p.d_a;
  const int64_t wv = static_cast<int64_t>(p.H) * p.dh;
  if (q_row_stride < wa || d_q_row_stride < wa) return set_err(SDM_RT_EINVAL, "q/d_q row stride < heads * addr_dim");
  if (dy_row_stride < wv) return set_err(SDM_RT_EINVAL, "dy_row_stride < heads * head_dim");
  if (!workspace || workspace_bytes < g.total)
    return set_err(SDM_RT_ENOSPACE, "workspace %zu bytes < required %zu", workspace_bytes, g.total);
  hipStream_t st = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  float* dw = reinterpret_cast<float*>(ws + g.off_dw);
  float* pf = reinterpret_cast<float*>(ws + g.off_pf);
  double* pd = reinterpret_cast<double*>(ws + g.off_pd);
  float* pk = reinterpret_cast<float*>(ws + g.off_pk);
  // 1. the value table gradient: picks sorted by (head, slot), summed by pieces, then the rows cut over several joined
  {
    int32_t* kin = reinterpret_cast<int32_t*>(ws + g.off_keys);
    int32_t* kout = kin + g.n_entries;
    int32_t* vin = kout + g.n_entries;
    int32_t* vout = vin + g.n_entries;
    int32_t* count = reinterpret_cast<int32_t*>(ws + g.off_count);
    int32_t* offsets = reinterpret_cast<int32_t*>(ws + g.off_offsets);
    const int n_keys = p.H * p.M + 1;
    hipLaunchKernelGGL(zero_i32_kernel, dim3(static_cast<unsigned>((n_keys + 255) / 256)), dim3(256), 0, st, count,
                       n_keys);
    if ((rc = check_launch("zero"))) return rc;
    hipLaunchKernelGGL(pick_keys_kernel, dim3(static_cast<unsigned>((g.n_entries + 255) / 256)), dim3(256), 0, st,
                       slots, g.n_entries, p.T, p.H, p.pitch, p.M, p.kk, kin, vin, count);
    if ((rc = check_launch("pick keys"))) return rc;
    size_t cb = g.cub_bytes;
    if (hipcub::DeviceScan::ExclusiveSum(ws + g.off_cub, cb, count, offsets, n_keys, st) != hipSuccess)
      return set_err(SDM_RT_ELAUNCH, "table backward: scan failed");
    cb = g.cub_bytes;
    if (hipcub::DeviceRadixSort::SortPairs(ws + g.off_cub, cb, kin, kout, vin, vout, static_cast<int>(g.n_entries), 0,
                                           g.key_bits, st) != hipSuccess)
      return set_err(SDM_RT_ELAUNCH, "table backward: sort failed");
    float* part = reinterpret_cast<float*>(ws + g.off_part);
    const unsigned sblocks = static_cast<unsigned>((values_pieces(g.n_entries) + 3) / 4);
    const bool vec = quad_rows(dy, dy_row_stride, dy_dtype);
#define SDM_RT_TV(DT, VEC)                                                                                          \
  hipLaunchKernelGGL((table_values_grad_kernel<DT, VEC>), dim3(sblocks), dim3(256), 0, st, kout, vout, offsets,     \
                     weights, static_cast<const DT*>(dy), dy_row_stride, d_values, part, p.T, p.H, p.pitch, p.M, p.dh)
    if (dy_dtype == SDM_RT_BF16) {
      if (vec) SDM_RT_TV(bf16_t, true); else SDM_RT_TV(bf16_t, false);
    } else {
      if (vec) SDM_RT_TV(float, true); else SDM_RT_TV(float, false);
    }
#undef SDM_RT_TV
    if ((rc = check_launch("table values grad"))) return rc;
    hipLaunchKernelGGL(table_values_join_kernel, dim3(static_cast<unsigned>((n_keys + 2) / 4)), dim3(256), 0, st,
                       offsets, count, part, d_values, p.H * p.M, p.dh);
    if ((rc = check_launch("table values join"))) return rc;
  }
  // 2. the per-pick gradients
  {
    const int64_t waves = static_cast<int64_t>(p.B) * p.T * p.H;
    const unsigned blocks = static_cast<unsigned>((waves + 3) / 4);
    const bool vec = quad_rows(dy, dy_row_stride, dy_dtype) && quad_rows(values, p.dh, values_dtype);
#define SDM_RT_TG_V(KP, VT, DT, VEC)                                                                                \
  hipLaunchKernelGGL((table_grad_kernel<KP, VT, DT, VEC>), dim3(blocks), dim3(256), 0, st, slots, weights,              \
                     static_cast<const VT*>(values), static_cast<const DT*>(dy), dy_row_stride, dw, p.B, p.T, p.H,  \
                     p.M, p.dh, p.kk)
#define SDM_RT_TG(KP, VT, DT) \
  if (vec) SDM_RT_TG_V(KP, VT, DT, true); else SDM_RT_TG_V(KP, VT, DT, false)
#define SDM_RT_TG_DT(KP, VT) \
  if (dy_dtype == SDM_RT_BF16) { SDM_RT_TG(KP, VT, bf16_t); } else { SDM_RT_TG(KP, VT, float); }
#define SDM_RT_TG_KP(VT) \
  if (p.pitch == 8) { SDM_RT_TG_DT(8, VT); } else { SDM_RT_TG_DT(16, VT); }
    if (values_dtype == SDM_RT_BF16) { SDM_RT_TG_KP(bf16_t); } else { SDM_RT_TG_KP(float); }
#undef SDM_RT_TG_KP
#undef SDM_RT_TG_DT
#undef SDM_RT_TG
#undef SDM_RT_TG_V
    if ((rc = check_launch("table grad"))) return rc;
  }
  // 3. softmax and product-key backward of the read set (no gate, no address bias)
  {
    GradPlan gp;
    gp.p = p;
    gp.n_blk = g.n_blk;
    gp.addr_waves = g.addr_waves;
    gp.tiles = g.tiles;
    AddrGradArgs a{};
    a.kz = q;
    a.kz_stride = q_row_stride;
    a.qz = q;
    a.qz_stride = q_row_stride;
    a.keys[0] = params->keys1;
    a.keys[1] = params->keys2;
    a.log_scale = params->log_scale;
    a.slot[1] = slots;
    a.wt[1] = weights;
    a.score[1] = scores;
    a.dot[1] = dw;
    a.n_cg = 1;
    a.dz[1] = d_q;
    a.dz_stride[1] = d_q_row_stride;
    a.part_f = pf;
    a.part_d = pd;
    a.part_k = pk;
    a.B = p.B;
    a.T = p.T;
    a.H = p.H;
    a.n_sub = p.n_sub;
    a.kk = p.kk;
    a.set0 = 1;
    rc = in_dtype == SDM_RT_BF16 ? by_half<AddrGradLaunch, bf16_t>(p.half, gp, a, st)
                                 : by_half<AddrGradLaunch, float>(p.half, gp, a, st);
    if (rc) return rc;
  }
  // 4. parameter sums
  GradSumsArgs a{};
  a.pk = pk;
  a.pf = pf;
  a.n_rec = g.n_blk;
  a.H = p.H;
  a.DA = p.d_a;
  a.n_sub = p.n_sub;
  a.half = p.half;
  a.keys[0] = params->keys1;
  a.keys[1] = params->keys2;
  a.log_scale = params->log_scale;
  a.d_keys[0] = d_keys1;
  a.d_keys[1] = d_keys2;
  a.d_log_scale = d_log_scale;
  return launch_grad_sums(a, st);
}

}  // extern "C"
