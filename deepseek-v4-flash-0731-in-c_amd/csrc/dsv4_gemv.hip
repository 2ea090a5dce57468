// dsv4_gemv.hip - decode-side kernels of the quantized MoE expert path for
// gfx950: activation FP8 quantisation, FP4/FP8 block-scaled GEMVs whose
// results are bit-identical to the reference's scalar loop order, the BF16
// router GEMV, the float-scale public GEMVs, dequantisers and the
// synthetic-checkpoint quantisers.
// The bit-exact GEMV row tiles are in dsv4_tiles.h.
#include <algorithm>

#include "dsv4_device.h"
#include "dsv4_gpu_internal.h"
#include "dsv4_tiles.h"

using namespace dsv4;

namespace dsv4 {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// ============================================================ activation ==
// One wave per 128-element group (src/dsv4/dsv4_model.c:5580-5606).
// grid = (ceil(n/128), nvec); x/qx rows are n apart, qscale rows ceil(n/128).
__global__ __launch_bounds__(64) void k_quant_fp8_act(float *__restrict__ qx,
                                                      float *__restrict__ qscale,
                                                      const float *__restrict__ x,
                                                      int n) {
  const int g = blockIdx.x, lane = threadIdx.x;
  const size_t row = blockIdx.y;
  const float *xr = x + row * (size_t)n;
  float *qr = qx + row * (size_t)n;
  const int base = g * 128;
  const int i0 = base + lane, i1 = base + 64 + lane;
  const float a = i0 < n ? xr[i0] : 0.0f;
  const float b = i1 < n ? xr[i1] : 0.0f;
  const float amax = wave_max(fmaxf(fabsf(a), fabsf(b)));
  const float scale = act_scale(amax);
  const float inv = 1.0f / scale;
  if (lane == 0) qscale[row * (size_t)((n + 127) / 128) + g] = scale;
  if (i0 < n) qr[i0] = quant_e4m3(a, inv);
  if (i1 < n) qr[i1] = quant_e4m3(b, inv);
}

// ============================================================== dequant ==
// FP4: out[r][c] = e2m1(W[r][c]) * e8m0(S[r][c/32]) (exact product).
__global__ void k_dequant_fp4(float *__restrict__ out, const uint8_t *__restrict__ W,
                              const uint8_t *__restrict__ S, int rows, int cols) {
  const size_t n = (size_t)rows * cols;
  const int pcols = (cols + 1) / 2, gcols = (cols + 31) / 32;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    const size_t r = i / cols, c = i % cols;
    const uint32_t b = W[r * pcols + (c >> 1)];
    const uint32_t nib = (c & 1) ? (b >> 4) : (b & 15u);
    out[i] = e2m1_decode(nib) * e8m0(S[r * gcols + c / 32]);
  }
}

// FP8: out[r][c] = e4m3(W[r][c]) * e8m0(S[r/128][c/128]).
__global__ void k_dequant_fp8(float *__restrict__ out, const uint8_t *__restrict__ W,
                              const uint8_t *__restrict__ S, int rows, int cols) {
  const size_t n = (size_t)rows * cols;
  const int cb = (cols + 127) / 128;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    const size_t r = i / cols, c = i % cols;
    out[i] = e4m3_decode(W[i]) * e8m0(S[(r / 128) * cb + c / 128]);
  }
}

// The FP4 GEMVs (dsv4_gemv_fp4_q / _pair_q / _batch_q,
// src/dsv4/dsv4_model.c:967-1380) on the decode layer's register tiles
// (dsv4_tiles.h): one (row, 32-column group) partial per lane as a sequential
// fmaf chain, one lane per row chaining the groups in order; NP
// passes per tile (paired: NP / 2 of each matrix over the same rows), every
// pass issued before the first FMA, NP chosen by the host so that one call
// spans about a thousand workgroups. The token's activation arrives as the
// E4M3 grid values the activation quant produced (floats): its codes are
// exact (e4m3_code) and go to LDS with the per-128 scales, loaded ahead of
// the weights. grid = (tiles, nvec); pair: y[0] / y[1] for W[0] / W[1].
template <int NP>
__global__ __launch_bounds__(256) void k_gemv_fp4_t(GemvArgs a, int pair) {
  extern __shared__ __align__(16) float lds[];
  __shared__ float s_y[256];
  const int tid = threadIdx.x, b = blockIdx.y;
  const Fp4Geom q = fp4_geom_np(a.in, NP);
  const int in = a.in;
  const float *qx = a.qx + (size_t)b * a.qx_stride;
  const float *qs = a.qscale + (size_t)b * a.qs_stride;
  // this thread's activation values (16 at 16 tid, and 4096 further for
  // in > 4096) and per-128 scale (thread i < in / 128: scale i), loaded
  // before the weights (loads complete in order: issued after the weights,
  // they would wait for every weight to land)
  const BufRsrc rx = buf_rsrc(qx, 4u * (uint32_t)in);
  uint4 xv[8];
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      xv[4 * k + i] = buf_load16(rx, 4u * (uint32_t)(16 * tid + 4096 * k) + 16u * i);
  const float qsv = buf_loadf(buf_rsrc(qs, 4u * (uint32_t)((in + 127) / 128)), 4u * (uint32_t)tid);
  Fp4RegsT<NP> R;
  const int half = q.tr / 2;
  const int r0 = pair ? blockIdx.x * half : blockIdx.x * q.tr;
  if (pair)
    fp4_pair_load(R, a.W[0], a.S[0], a.W[1], a.S[1], in, a.rows, r0, q);
  else
    fp4_tile_load(R, a.W[0], a.S[0], in, a.rows, r0, q);
  uint8_t *cl = reinterpret_cast<uint8_t *>(lds) + (size_t)q.tr * pair_stride(q.G) * 8;
  uint8_t *x8 = cl + 4096;
  float *xs = reinterpret_cast<float *>(x8 + ((in + 15) & ~15));
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int base = 16 * tid + 4096 * k;
    if (base < in) {
      uint32_t c[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint4 v = xv[4 * k + i];
        c[i] = e4m3_code(u2f(v.x)) | (e4m3_code(u2f(v.y)) << 8) |
               (e4m3_code(u2f(v.z)) << 16) | (e4m3_code(u2f(v.w)) << 24);
      }
      *reinterpret_cast<uint4 *>(x8 + base) = make_uint4(c[0], c[1], c[2], c[3]);
    }
  }
  if (tid < (in + 127) / 128) xs[tid] = qsv;  // in <= 8192: at most 64 scales
  __syncthreads();
  fp4_tile_x_lds(R, x8, xs, q);
  float2 *ps = reinterpret_cast<float2 *>(lds);
  if (pair) {
    fp4_pair_finish(R, s_y, a.rows, r0, q, ps, cl);
    __syncthreads();
    if (a.swi_y) {  // routed_swiglu_quant's y (src/dsv4/dsv4_model.c:6258-6268)
      if (tid < half && r0 + tid < a.rows)
        a.swi_y[(size_t)b * a.y_stride + r0 + tid] =
            bf16_round(swiglu_t(s_y[tid], s_y[tid + half], a.swi_limit) *
                       (a.swi_w ? *a.swi_w : 1.0f));
    } else if (tid < q.tr && r0 + tid % half < a.rows) {
      a.y[tid / half][(size_t)b * a.y_stride + r0 + tid % half] = s_y[tid];
    }
  } else {
    fp4_tile_finish(R, a.y[0] + (size_t)b * a.y_stride, a.rows, r0, q, ps, cl);
  }
}

// ========================================================= FP8 GEMV =====
// dsv4_gemv_fp8_q / _pair_q / _batch_q (src/dsv4/dsv4_model.c:571-961) for
// any width up to 8192 and any number of token vectors, bit-exact: per
// (row, 128-column block) a 128-long sequential fmaf chain, then per row the
// block chain acc = fmaf(p, qscale * ws, acc) in order (NaN block scale:
// the block is skipped, as in the reference).
//
// Lane t of a workgroup is (row t / SL, slot t % SL) and owns blocks slot
// and slot + SL; SL (8, 16 or 32 lanes per row) is the smallest that leaves
// every lane at most two blocks, so a lane's whole weight slice (2 x 128 B)
// is loaded into registers before any arithmetic and the workgroup's rows
// stream from HBM in one go. Tokens are taken G at a time: each 16-column
// piece is decoded once and feeds G chains, and the weights stay in
// registers across all the token groups, so a batch reads them from HBM
// once. LDS: the G tokens' activations (padded to 132 floats per block) and
// their scales, and the (partial, scale) pairs of the block chains.
template <int SL, int G>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(G == 4 ? 4 : 1))) void k_fp8_proj(
    GemvArgs a, int nvec, int gpw, int vec4) {
  constexpr int TR = 256 / SL;
  extern __shared__ __align__(16) float lds[];
  const int m = blockIdx.z, t = threadIdx.x, lr = t / SL, slot = t % SL;
  const int in = a.in, rows = a.rows, r0 = blockIdx.x * TR;
  const int CB = (in + 127) / 128, stride = pair_stride(CB);
  float *xs = lds;                                   // [G][CB][132]
  float *qs = xs + (size_t)G * CB * 132;             // [G][CB]
  float2 *ps = reinterpret_cast<float2 *>(qs + ((G * CB + 3) & ~3));  // [G][TR][stride]
  // per wave: the exchange of its rows' weights (64 chunks of 128 B, 144 B
  // apart), over the space of xs, qs and ps before they are written
  uint8_t *xch = reinterpret_cast<uint8_t *>(lds) + (t / 64) * 9216;

  // this workgroup's token groups: gpw groups of G from blockIdx.y * gpw
  const int tbeg = blockIdx.y * gpw * G, tend = min(nvec, tbeg + gpw * G);
  // the first group's activations (up to 8192 values) are loaded ahead of the
  // weights: loads complete in order, so behind the weights they would wait
  // for every weight to land
  const bool xpre = vec4 && G * in <= 8192;  // then also G CB <= 256 scales
  float4 xr[8];
  float qr = 0.0f;
  if (xpre) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int i = 4 * t + 1024 * k;
      const int g = i / in, c = i % in;
      xr[k] = i < G * in && tbeg + g < nvec
                  ? *reinterpret_cast<const float4 *>(a.qx + (size_t)(tbeg + g) * a.qx_stride + c)
                  : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    if (t < G * CB && tbeg + t / CB < nvec)
      qr = a.qscale[(size_t)(tbeg + t / CB) * a.qs_stride + t % CB];
  }

  // the weights (zeros past the matrix): round j covers the row's columns
  // [128 SL j, 128 SL (j + 1)); load i of the SL lanes of a row reads 16 SL
  // contiguous bytes (chunk i SL + slot of the round), so every load
  // instruction covers whole lines; the chunks then go through the wave's
  // LDS region to the lane that owns their block (block slot + SL j)
  const uint32_t nrow = (uint32_t)max(0, min(TR, rows - r0));
  const BufRsrc rw = buf_rsrc(a.W[m] + (size_t)r0 * in, nrow * (uint32_t)in);
  const BufRsrc rs = buf_rsrc(a.S[m], (uint32_t)((rows + 127) / 128) * CB);
  uint4 w[16];
  uint32_t sc[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const uint32_t cb = (uint32_t)(slot + SL * j);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t c = (uint32_t)(SL * 128 * j + 16 * (SL * i + slot));
      w[8 * j + i] = buf_load16(rw, c < (uint32_t)in ? (uint32_t)lr * (uint32_t)in + c
                                                     : 0xFFFFFFF0u);
    }
    sc[j] = __builtin_amdgcn_raw_buffer_load_b8(
        rs, cb < (uint32_t)CB && (uint32_t)lr < nrow ? (uint32_t)((r0 + lr) / 128) * CB + cb
                                                      : 0xFFFFFFF0u, 0, 0);
  }
  {
    // the exchange: chunk q = SL i + slot of round j lies in block q / 8 at
    // piece q % 8; the wave's rows (lr % (64 / SL)) are SL 144 B apart
    const int wr = lr % (64 / SL);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (SL * 128 * j >= in) break;  // a round wholly past the row (uniform)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int q = SL * i + slot;
        *reinterpret_cast<uint4 *>(xch + (wr * SL + q / 8) * 144 + (q % 8) * 16) = w[8 * j + i];
      }
      __builtin_amdgcn_wave_barrier();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < 8; ++i)
        w[8 * j + i] = *reinterpret_cast<const uint4 *>(xch + (wr * SL + slot) * 144 + 16 * i);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_wave_barrier();
    }
  }
  __syncthreads();  // every wave's exchange read before xs, qs and ps take the space
  if (xpre) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int i = 4 * t + 1024 * k;
      const int g = i / in, c = i % in;
      if (i < G * in)
        *reinterpret_cast<float4 *>(xs + (size_t)g * CB * 132 + (c / 128) * 132 + (c % 128)) =
            xr[k];
    }
    if (t < G * CB) qs[t] = qr;
  }

  for (int t0 = tbeg; t0 < tend; t0 += G) {
    // the group's activations and scales into LDS (zeros past the last token)
    if (xpre && t0 == tbeg) {
      // loaded ahead of the weights
    } else if (vec4) {
      for (int i = 4 * t; i < G * in; i += 1024) {
        const int g = i / in, c = i % in;
        const float4 v = t0 + g < nvec
                             ? *reinterpret_cast<const float4 *>(
                                   a.qx + (size_t)(t0 + g) * a.qx_stride + c)
                             : make_float4(0.f, 0.f, 0.f, 0.f);
        *reinterpret_cast<float4 *>(xs + (size_t)g * CB * 132 + (c / 128) * 132 + (c % 128)) = v;
      }
    } else {
      for (int i = t; i < G * in; i += 256) {
        const int g = i / in, c = i % in;
        xs[(size_t)g * CB * 132 + (c / 128) * 132 + (c % 128)] =
            t0 + g < nvec ? a.qx[(size_t)(t0 + g) * a.qx_stride + c] : 0.0f;
      }
    }
    if (!(xpre && t0 == tbeg))
      for (int i = t; i < G * CB; i += 256) {
        const int g = i / CB;
        qs[i] = t0 + g < nvec ? a.qscale[(size_t)(t0 + g) * a.qs_stride + i % CB] : 0.0f;
      }
    __syncthreads();
    if (r0 + lr < rows) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int cb = slot + SL * j;
        if (cb < CB) {
          const int len = min(128, in - cb * 128);
          float part[G];
#pragma unroll
          for (int g = 0; g < G; ++g) part[g] = 0.0f;
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            if (16 * i < len) {
              const uint32_t wd[4] = {w[8 * j + i].x, w[8 * j + i].y, w[8 * j + i].z,
                                      w[8 * j + i].w};
              float v[16];
#pragma unroll
              for (int d = 0; d < 4; ++d) {
                const float2 lo = fp8x2<false>(wd[d]), hi = fp8x2<true>(wd[d]);
                v[4 * d] = lo.x;
                v[4 * d + 1] = lo.y;
                v[4 * d + 2] = hi.x;
                v[4 * d + 3] = hi.y;
              }
#pragma unroll
              for (int g = 0; g < G; ++g) {
                const float *xb = xs + (size_t)g * CB * 132 + cb * 132 + 16 * i;
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                  const float4 xv = *reinterpret_cast<const float4 *>(xb + 4 * d);
                  part[g] = fmaf(v[4 * d], xv.x, part[g]);
                  part[g] = fmaf(v[4 * d + 1], xv.y, part[g]);
                  part[g] = fmaf(v[4 * d + 2], xv.z, part[g]);
                  part[g] = fmaf(v[4 * d + 3], xv.w, part[g]);
                }
              }
            }
          }
#pragma unroll
          for (int g = 0; g < G; ++g) {
            float s = qs[g * CB + cb] * e8m0(sc[j]);
            float p = part[g];
            if (sc[j] == 255u) {  // NaN scale: the reference skips the block
              p = 0.0f;
              s = 0.0f;
            }
            ps[(size_t)(g * TR + lr) * stride + cb] = make_float2(p, s);
          }
        }
      }
    }
    __syncthreads();
    if (t < G * TR) {
      const int g = t / TR, r = t % TR;
      if (r0 + r < rows && t0 + g < nvec) {
        const float acc = pair_chain(ps + (size_t)(g * TR + r) * stride, CB);
        a.y[m][(size_t)(t0 + g) * a.y_stride + r0 + r] = a.round_out ? bf16_round(acc) : acc;
      }
    }
    __syncthreads();  // LDS is refilled by the next group
  }
}

// Several tokens on the fp32 matrix unit: an MFMA 16x16x4 adds its four
// products in column order, each as one rounded fma (k_bf16_rows_mfma), so a
// tile started from zero at every 128-column block runs the block's chains of
// 16 rows x 16 tokens bit for bit. Every block's partials go to LDS, and a
// thread per (row, token) chains the (partial, scale) pairs in order, so the
// blocks are independent: KS waves share a row tile (wave k: blocks k, k + KS,
// ...) where the rows alone leave SIMDs idle (4096 rows: 256 tiles), 4 / KS
// tiles per workgroup. Each wave stages for itself, without barriers (its LDS
// operations are in order): a lane loads 16 consecutive columns of a row and
// of a token, FM_D steps of 64 columns ahead, writes them to LDS widened and
// split by c % 4 (a choice of registers) and reads its column of 16 back with
// one 16-byte read, the next step's while this step's MFMAs run. Bound: the
// MFMA's latency where a SIMD has one wave, then the matrix rate, on tokens
// padded to 16. in a multiple of 128. Token groups of one row tile are
// neighbours on one XCD: its weights come from that L2 after the first.
#define FM_D 4
template <int KS>
static size_t fp8_mfma_lds(int CB) {
  return ((size_t)4 * 2 * 16 * MT_RS + (size_t)(4 / KS) * CB * 257 + (size_t)CB * 16) * 4;
}

template <int KS>
__global__ __launch_bounds__(256) void k_fp8_proj_mfma(GemvArgs a, int nvec, int units,
                                                       int groups) {
  constexpr int NT = 4 / KS;  // row tiles per workgroup
  extern __shared__ __align__(16) float lds[];
  const int tid = threadIdx.x, l = tid & 63, l16 = l & 15, g = l >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), tl = wave / KS, ks = wave % KS;
  const int mat = blockIdx.z, in = a.in, CB = in / 128;
  const int k8 = blockIdx.x >> 3;
  const int unit = (k8 / groups) * 8 + (blockIdx.x & 7), t0 = (k8 % groups) * 16;
  if (unit >= units) return;
  const int r0 = unit * 16 * NT, nt = min(16, nvec - t0);
  float *lw = lds + wave * 2 * 16 * MT_RS, *lx = lw + 16 * MT_RS;
  float *parts = lds + 4 * 2 * 16 * MT_RS;                    // [NT][CB][256]
  float *sq = parts + (size_t)NT * CB * 256;                  // [CB][16]
  uint32_t *sw = reinterpret_cast<uint32_t *>(sq + CB * 16);  // [NT][CB]
  const int wr0 = r0 + 16 * tl;  // this wave's rows
  const int nrow = __builtin_amdgcn_readfirstlane(max(0, min(16, a.rows - wr0)));
  const BufRsrc rw = buf_rsrc(a.W[mat] + (size_t)wr0 * in, (uint32_t)nrow * (uint32_t)in);
  const BufRsrc rx = buf_rsrc(a.qx + (size_t)t0 * a.qx_stride,
                              4u * ((uint32_t)(nt - 1) * (uint32_t)a.qx_stride + (uint32_t)in));
  // lane = (row l / 4, columns 16 (l % 4) .. + 15 of a step); rows past the
  // matrix or the tokens are out of range (zeros), blocks past the width not
  // stored
  const uint32_t wo = (uint32_t)(l >> 2) * (uint32_t)in + 16u * (uint32_t)(l & 3);
  const uint32_t xo = (l >> 2) < nt ? 4u * (uint32_t)(l >> 2) * (uint32_t)a.qx_stride +
                                          64u * (uint32_t)(l & 3)
                                    : 0x80000000u;
  const int po = mt_at(l >> 2, l & 3);
  const int ro[4] = {mt_at(l16, 0) + 16 * g, mt_at(l16, 1) + 16 * g, mt_at(l16, 2) + 16 * g,
                     mt_at(l16, 3) + 16 * g};
  uint4 W[FM_D], X[FM_D][4];
  auto load = [&](int d, int i) {  // step i: half i % 2 of block ks + KS (i / 2)
    const uint32_t c = 128u * (uint32_t)(ks + KS * (i >> 1)) + 64u * (uint32_t)(i & 1);
    W[d] = buf_load16(rw, wo + c);
#pragma unroll
    for (int q = 0; q < 4; ++q) X[d][q] = buf_load16(rx, xo + 4u * c + 16u * q);
  };
  auto put = [&](int d) {
    const uint32_t wd[4] = {W[d].x, W[d].y, W[d].z, W[d].w};
    float2 lo[4], hi[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      lo[q] = fp8x2<false>(wd[q]);
      hi[q] = fp8x2<true>(wd[q]);
    }
    *reinterpret_cast<float4 *>(lw + po) = make_float4(lo[0].x, lo[1].x, lo[2].x, lo[3].x);
    *reinterpret_cast<float4 *>(lw + po + 16) = make_float4(lo[0].y, lo[1].y, lo[2].y, lo[3].y);
    *reinterpret_cast<float4 *>(lw + po + 32) = make_float4(hi[0].x, hi[1].x, hi[2].x, hi[3].x);
    *reinterpret_cast<float4 *>(lw + po + 48) = make_float4(hi[0].y, hi[1].y, hi[2].y, hi[3].y);
    const uint4 *c = X[d];
    *reinterpret_cast<uint4 *>(lx + po) = make_uint4(c[0].x, c[1].x, c[2].x, c[3].x);
    *reinterpret_cast<uint4 *>(lx + po + 16) = make_uint4(c[0].y, c[1].y, c[2].y, c[3].y);
    *reinterpret_cast<uint4 *>(lx + po + 32) = make_uint4(c[0].z, c[1].z, c[2].z, c[3].z);
    *reinterpret_cast<uint4 *>(lx + po + 48) = make_uint4(c[0].w, c[1].w, c[2].w, c[3].w);
  };
  f32x4 av[2][4], bv[2][4];
  auto get = [&](int o) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      av[o][q] = *reinterpret_cast<const f32x4 *>(lw + ro[q]);
      bv[o][q] = *reinterpret_cast<const f32x4 *>(lx + ro[q]);
    }
  };
#pragma unroll
  for (int d = 0; d < FM_D; ++d) load(d, d);
  for (int i = tid; i < CB * 16; i += 256) {
    const int t = i & 15;
    sq[i] = t < nt ? a.qscale[(size_t)(t0 + t) * a.qs_stride + (i >> 4)] : 0.0f;
  }
  for (int i = tid; i < NT * CB; i += 256) {
    const int r = min(r0 + 16 * (i / CB), a.rows - 1);
    sw[i] = a.S[mat][(size_t)(r / 128) * CB + i % CB];
  }
  put(0);
  load(0, FM_D);
  get(0);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int i0 = 0; ks + KS * (i0 >> 1) < CB; i0 += FM_D) {
#pragma unroll
    for (int d = 0; d < FM_D; ++d) {
      // the next step into LDS and its operands out of it, its registers
      // reloaded, beside the MFMAs of step i0 + d
      const int nd = (d + 1) % FM_D;
      put(nd);
      load(nd, i0 + d + 1 + FM_D);
      get((d + 1) % 2);
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av[d % 2][q][e], bv[d % 2][q][e], acc, 0, 0,
                                                     0);
      // one MFMA, then what fits into its shadow
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
        __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // LDS write
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // load
        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);  // VALU
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
        __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (d % 2) {  // the block's end
        const int cb = ks + KS * ((i0 + d) >> 1);
        if (cb < CB)  // uniform
          *reinterpret_cast<f32x4 *>(parts + ((size_t)tl * CB + cb) * 256 + 16 * l16 + 4 * g) =
              acc;
        acc = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
  }
  __syncthreads();
  // thread i: row i % 16 of the tile, token i / 16
  const int tok = tid >> 4;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int row = r0 + 16 * t + (tid & 15);
    if (row >= a.rows || tok >= nt) continue;
    float o = 0.0f;
#pragma unroll 8
    for (int cb = 0; cb < CB; ++cb) {
      const uint32_t sc = sw[t * CB + cb];
      const float n =
          fmaf(parts[((size_t)t * CB + cb) * 256 + tid], sq[cb * 16 + tok] * e8m0(sc), o);
      o = sc == 255u ? o : n;  // NaN scale: the reference skips the block
    }
    a.y[mat][(size_t)(t0 + tok) * a.y_stride + row] = a.round_out ? bf16_round(o) : o;
  }
}

template <int KS>
static int launch_fp8_proj_mfma(const GemvArgs *a, int nvec, int nmat, hipStream_t st) {
  const int CB = a->in / 128, rt = 16 * (4 / KS);
  const int units = (a->rows + rt - 1) / rt, groups = (nvec + 15) / 16;
  const size_t lds = fp8_mfma_lds<KS>(CB);
  if (lds > 64 * 1024)  // (a host-side setting of the kernel)
    DSV4G_HIP(hipFuncSetAttribute((const void *)k_fp8_proj_mfma<KS>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)(140 * 1024)));
  hipLaunchKernelGGL(k_fp8_proj_mfma<KS>, dim3((units + 7) / 8 * 8 * groups, 1, nmat), dim3(256),
                     lds, st, *a, nvec, units, groups);
  return 0;
}

// Token groups per workgroup: all of them when the row tiles alone give
// 1024 or more workgroups (each weight read from HBM once); otherwise the
// groups are spread so the launch still has about that many (a small
// matrix's re-reads come from the caches).
static size_t max_size(size_t a, size_t b) { return a > b ? a : b; }

template <int SL, int G>
static void launch_fp8_proj(const GemvArgs *a, int nvec, int nmat, hipStream_t st) {
  constexpr int TR = 256 / SL;
  const int CB = (a->in + 127) / 128;
  // xs, qs and ps, or the four waves' weight exchanges before them
  const size_t lds = max_size(((size_t)G * CB * 132 + ((G * CB + 3) & ~3)) * 4 +
                                  (size_t)G * TR * pair_stride(CB) * 8,
                              (size_t)4 * 9216);
  const int tiles = (a->rows + TR - 1) / TR * nmat, groups = (nvec + G - 1) / G;
  const int split = min(groups, max(1, 1024 / tiles));
  const int gpw = (groups + split - 1) / split;
  const int vec4 = ((uintptr_t)a->qx % 16 == 0) && (a->qx_stride % 4 == 0);
  hipLaunchKernelGGL((k_fp8_proj<SL, G>),
                     dim3((a->rows + TR - 1) / TR, (groups + gpw - 1) / gpw, nmat), dim3(256),
                     lds, st, *a, nvec, gpw, vec4);
}

// ======================================================== BF16 GEMV =====
// y[r] = the reference's column-order chain acc = fmaf(bf16(W[r][c]), x[c],
// acc) (src/dsv4/dsv4_model.c:298-303; its 8-row AVX2 path runs the same
// chain per row): one lane per (row, token), the row read 16 bytes at a
// time, x shared by the wave (one line per load). Bit-exact; the cost is
// one dependent fmaf per column.
__global__ __launch_bounds__(64) void k_gemv_bf16(float *__restrict__ y,
                                                  const float *__restrict__ x,
                                                  const uint16_t *__restrict__ W, int in,
                                                  int out, int round_out, size_t y_stride,
                                                  size_t x_stride) {
  const int row = blockIdx.x * 64 + threadIdx.x;
  const int b = blockIdx.y;
  if (row >= out) return;
  const float *xb = x + (size_t)b * x_stride;
  const uint16_t *wr = W + (size_t)row * in;
  float acc = 0.0f;
  int c = 0;
  if ((in & 7) == 0) {
    for (; c < in; c += 8) {
      const uint4 w = *reinterpret_cast<const uint4 *>(wr + c);
      const uint32_t wd[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        acc = fmaf(u2f(wd[d] << 16), xb[c + 2 * d], acc);
        acc = fmaf(u2f(wd[d] & 0xFFFF0000u), xb[c + 2 * d + 1], acc);
      }
    }
  }
  for (; c < in; ++c) acc = fmaf(bf16_to_f32(wr[c]), xb[c], acc);
  y[(size_t)b * y_stride + row] = round_out ? bf16_round(acc) : acc;
}

// ====================================================== row chains =====
// The same chains, one lane per output row, for rows whose bytes are a
// multiple of 16: each lane reads its own row straight from HBM 16 bytes at
// a time through one buffer range over the wave's 64 rows (a row past the
// matrix reads zeros), 16 loads per chunk and two chunks in turn, so 32
// loads (512 bytes of the row) are in flight while a chunk is chained; x
// (every token, at most RC_XBYTES) and the FP8 block scales of the wave's
// row blocks are staged in LDS once and read as broadcasts. The per-column arithmetic is the reference's, so the results
// are bit for bit those of the one-load-at-a-time kernels above; they only
// wait less.
//   RC_BF16: acc_t = fmaf(bf16(w), x_t[c], acc_t) for MAXB tokens at most
//            (dsv4_gemv_bf16(_batch), src/dsv4/dsv4_model.c:266-367; the vocab
//            head's head_logits_block, :7221-7255);
//   RC_FP8_X: acc += w * (x * s)   (dsv4_gemv_fp8, src/dsv4/dsv4_ops.c:176-209);
//   RC_FP8_XS: the same when the wave's 64 rows share one row block (block a
//            multiple of 64): xs = x * s is formed once per column in LDS,
//            as the reference forms it once per row block;
//   RC_FP8_T: acc += (w * x) * s   (dsv4_gemv_fp8_tbl, :216-239),
// unfused as the reference is built; s = wscale[row / block][c / block],
// block a multiple of 16.
#define RC_BF16 0
#define RC_FP8_X 1
#define RC_FP8_T 2
#define RC_FP8_XS 3
#define RC_CHUNK 16           // 16-byte loads per chunk
#define RC_XBYTES (64 * 1024)  // LDS for x

struct RowChainArgs {
  float *y;
  const float *x;
  const uint8_t *W;
  const float *wscale;
  int in, rows, block, batch, round_out;
  size_t y_stride, x_stride;
};

// Pieces byte0, byte0 + 16, ... of the lane's row (at row_off in the
// wave's range; live: the lane has a row). Past the row, or without one:
// zeros, nothing read.
__device__ __forceinline__ void rc_load(uint4 (&w)[RC_CHUNK], BufRsrc r, uint32_t row_off,
                                        bool live, uint32_t byte0, uint32_t rb) {
#pragma unroll
  for (int i = 0; i < RC_CHUNK; ++i) {
    const uint32_t b = byte0 + 16u * i;
    w[i] = buf_load16(r, live && b < rb ? row_off + b : 0xFFFFFFF0u);
  }
}

// One chunk: columns c0 .. of the 16-byte pieces w (8 BF16 or 16 FP8 each);
// xs: x in LDS, token t at t * in.
template <int KIND, int MAXB>
__device__ __forceinline__ void rc_chain(const RowChainArgs &a, const uint4 (&w)[RC_CHUNK],
                                         int c0, float (&acc)[MAXB], const float *srow,
                                         const float *xs) {
  constexpr int CPP = KIND == RC_BF16 ? 8 : 16;  // columns per piece
#pragma unroll
  for (int i = 0; i < RC_CHUNK; ++i) {
    const int c = c0 + CPP * i;
    if (c >= a.in) break;  // uniform: the chunk's last pieces may lie past the row
    const uint32_t wd[4] = {w[i].x, w[i].y, w[i].z, w[i].w};
    if (KIND == RC_BF16) {
#pragma unroll
      for (int t = 0; t < MAXB; ++t) {
        if (t >= a.batch) break;
        const float4 *xt = reinterpret_cast<const float4 *>(xs + (size_t)t * a.in + c);
        const float4 x0 = xt[0], x1 = xt[1];
        const float xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          acc[t] = fmaf(u2f(wd[d] << 16), xv[2 * d], acc[t]);
          acc[t] = fmaf(u2f(wd[d] & 0xFFFF0000u), xv[2 * d + 1], acc[t]);
        }
      }
    } else if (KIND == RC_FP8_XS) {
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const float2 lo = fp8x2<false>(wd[d]), hi = fp8x2<true>(wd[d]);
        const float wv[4] = {lo.x, lo.y, hi.x, hi.y};
        const float4 x4 = *reinterpret_cast<const float4 *>(xs + c + 4 * d);
        const float xv[4] = {x4.x, x4.y, x4.z, x4.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[0] += wv[e] * xv[e];
      }
    } else {
      const float s = srow[c / a.block];
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const float2 lo = fp8x2<false>(wd[d]), hi = fp8x2<true>(wd[d]);
        const float wv[4] = {lo.x, lo.y, hi.x, hi.y};
        const float4 x4 = *reinterpret_cast<const float4 *>(xs + c + 4 * d);
        const float xv[4] = {x4.x, x4.y, x4.z, x4.w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[0] += KIND == RC_FP8_X ? wv[e] * (xv[e] * s) : (wv[e] * xv[e]) * s;
      }
    }
  }
}

template <int KIND, int MAXB>
__global__ __launch_bounds__(64) void k_rowchain(RowChainArgs a) {
  extern __shared__ __align__(16) float xs[];  // batch * in floats
  const int r0 = blockIdx.x * 64, lane = threadIdx.x, row = r0 + lane;
  for (int t = 0; t < a.batch; ++t)
    for (int i = lane; i < a.in / 4; i += 64)
      reinterpret_cast<float4 *>(xs + (size_t)t * a.in)[i] =
          reinterpret_cast<const float4 *>(a.x + (size_t)t * a.x_stride)[i];
  const uint32_t rb = (uint32_t)a.in * (KIND == RC_BF16 ? 2u : 1u);
  const int nrow = min(64, a.rows - r0);
  const BufRsrc r = buf_rsrc(a.W + (size_t)r0 * rb, (uint32_t)nrow * rb);
  const bool live = lane < nrow;
  const uint32_t row_off = (uint32_t)lane * rb;
  const float *srow = nullptr;
  if (KIND == RC_FP8_XS) {
    // xs[c] = x[c] * s[row block][c / block], the row block of all 64 rows
    const int cblocks = (a.in + a.block - 1) / a.block;
    const float *s = a.wscale + (size_t)(r0 / a.block) * cblocks;
    __syncthreads();  // x in LDS
    for (int i = lane; i < a.in; i += 64) xs[i] = xs[i] * s[i / a.block];
  } else if (KIND != RC_BF16) {
    // the block scales of the wave's row blocks, after x in LDS
    const int cblocks = (a.in + a.block - 1) / a.block;
    const int rb0 = r0 / a.block, nrb = (min(r0 + 63, a.rows - 1)) / a.block - rb0 + 1;
    float *sc = xs + (size_t)a.batch * a.in;
    for (int i = lane; i < nrb * cblocks; i += 64)
      sc[i] = a.wscale[(size_t)rb0 * cblocks + i];
    srow = sc + (size_t)(min(row, a.rows - 1) / a.block - rb0) * cblocks;
  }
  float acc[MAXB];
#pragma unroll
  for (int t = 0; t < MAXB; ++t) acc[t] = 0.0f;
  constexpr uint32_t CB = 16u * RC_CHUNK;  // bytes per chunk
  constexpr int CPC = (KIND == RC_BF16 ? 8 : 16) * RC_CHUNK;  // columns per chunk
  uint4 A[RC_CHUNK], B[RC_CHUNK];
  rc_load(A, r, row_off, live, 0, rb);
  __syncthreads();  // x in LDS
  for (uint32_t b0 = 0; b0 < rb; b0 += 2 * CB) {
    const int c0 = (int)(b0 / CB) * CPC;
    rc_load(B, r, row_off, live, b0 + CB, rb);
    rc_chain<KIND, MAXB>(a, A, c0, acc, srow, xs);
    rc_load(A, r, row_off, live, b0 + 2 * CB, rb);
    rc_chain<KIND, MAXB>(a, B, c0 + CPC, acc, srow, xs);
  }
  if (row >= a.rows) return;
#pragma unroll
  for (int t = 0; t < MAXB; ++t) {
    if (t >= a.batch) break;
    a.y[(size_t)t * a.y_stride + row] = a.round_out ? bf16_round(acc[t]) : acc[t];
  }
}

// ================================================ product chains (FP8) ===
// dsv4_gemv_fp8 / dsv4_gemv_fp8_tbl with the products formed apart from the
// chain. The reference's per-row loop acc += p[c] (p[c] = w[c] * xs[c] with
// xs = x * s, or (w[c] * x[c]) * s; each product rounded on its own, the
// build unfused; src/dsv4/dsv4_ops.c:176-239) adds products that do not
// depend on acc. So all four waves of a workgroup form its PC_ROWS rows'
// products into LDS (rows padded by 16 bytes, so that the chain lanes'
// reads of one column fall in distinct banks), and then one lane per row
// runs only the dependent adds, in column order, four products per LDS read
// and the next 32 products' reads in flight while 32 are added. (One lane
// per row decoding, scaling, multiplying and adding every column ran at
// about 23 cycles per column; an add chain alone runs at its dependency
// latency.) The rows of a workgroup share one row block (block a multiple of
// 16); in a multiple of 32, at most PC_MAXIN.
#define PC_ROWS 8
#define PC_MAXIN 2048

// acc + p[0] + ... + p[4 N4 - 1] in order, p in LDS (16-byte aligned): fully
// unrolled, so every read is one instruction with an immediate offset and
// the lane's instruction stream holds nothing but reads and the dependent
// adds (in a single wave every other instruction delays the chain by its
// issue time). The reads run PC_LA float4 ahead of the adds in a register
// ring; an empty asm on acc after each float4's adds pins that order (left
// to itself the compiler keeps only one or two reads in flight).
#define PC_LA 7
template <int N4>
__device__ __forceinline__ float pc_chain_fixed(const float4 *p4, float acc) {
  constexpr int LA = N4 < PC_LA ? N4 : PC_LA, R = LA + 1;
  float4 v[R];
#pragma unroll
  for (int j = 0; j < LA; ++j) v[j] = p4[j];
#pragma unroll
  for (int j = 0; j < N4; ++j) {
    if (j + LA < N4) v[(j + LA) % R] = p4[j + LA];
    const float4 c = v[j % R];
    acc = acc + c.x;
    acc = acc + c.y;
    acc = acc + c.z;
    acc = acc + c.w;
    asm volatile("" : "+v"(acc)::"memory");
  }
  return acc;
}

// The products of piece k of the calling thread (16 columns of one row) into
// the row's LDS products: p = w * xs (MODE 0) or (w * x) * s (MODE 1).
template <int MODE>
__device__ __forceinline__ void pc_products(const uint4 w, int r, int c, const float *xs,
                                            const float *srow, int block, int ps, float *pr) {
  const uint32_t wd[4] = {w.x, w.y, w.z, w.w};
  const float sc = MODE == 1 ? srow[c / block] : 1.0f;
  float4 *dst = reinterpret_cast<float4 *>(pr + (size_t)r * ps + c);
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const float2 lo = fp8x2<false>(wd[d]), hi = fp8x2<true>(wd[d]);
    const float4 xv = *reinterpret_cast<const float4 *>(xs + c + 4 * d);
    float4 p;
    if (MODE == 0) {
      p = make_float4(lo.x * xv.x, lo.y * xv.y, hi.x * xv.z, hi.y * xv.w);
    } else {
      p = make_float4((lo.x * xv.x) * sc, (lo.y * xv.y) * sc, (hi.x * xv.z) * sc,
                      (hi.y * xv.w) * sc);
    }
    dst[d] = p;
  }
}

// x is loaded first (its loads would otherwise wait behind every weight load:
// the memory counter is in order), staged as x or x * s, then waves 1-3 form
// every product as their weight loads land, in column order: load k of a
// producer lane is piece (tid - 64) + 192 k, that is row i % PC_ROWS of the
// 16-column chunk i / PC_ROWS, so load k covers columns [384 k, 384 k + 384)
// of all rows; after its products of load k a producer wave counts itself in
// s_cnt[k]. Wave 0's chain lanes start as soon as the first 384 columns are
// counted and check a count only when the chain reaches a load not yet seen
// complete; so the chain starts after one load round trip, not half the row.
#define PC_LOADS ((PC_ROWS * PC_MAXIN / 16 + 191) / 192)  // weight loads per producer lane
#define PC_XQ (PC_MAXIN / 4 / 256)                         // x float4 per thread
template <int MODE>
__global__ __launch_bounds__(256) void k_fp8_prodchain(float *__restrict__ y,
                                                       const float *__restrict__ x,
                                                       const uint8_t *__restrict__ W,
                                                       const float *__restrict__ wscale, int in,
                                                       int rows, int block) {
  extern __shared__ __align__(16) float lds[];
  __shared__ int s_cnt[PC_LOADS];
  const int tid = threadIdx.x, wave = tid >> 6, r0 = blockIdx.x * PC_ROWS;
  const int cblocks = (in + block - 1) / block;
  const int ps = in + 4;             // product row stride (floats)
  float *xs = lds;                   // [in] x (MODE 1) or x * s (MODE 0)
  float *pr = lds + in;              // [PC_ROWS][ps] products
  float *ss = pr + PC_ROWS * ps;     // [cblocks] the row block's scales
  const float *srow = wscale + (size_t)(r0 / block) * cblocks;
  const int npiece = PC_ROWS * (in / 16);
  const int nrow = min(PC_ROWS, rows - r0);
  // the scales and x are loaded before the weights: a wait for them then
  // leaves the weight loads in flight (the memory counter is in order)
  const float sv = tid < cblocks ? srow[tid] : 0.0f;
  float4 xv[PC_XQ];
#pragma unroll
  for (int q = 0; q < PC_XQ; ++q) {
    const int i = tid + 256 * q;
    xv[q] = i < in / 4 ? reinterpret_cast<const float4 *>(x)[i] : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  const BufRsrc rw = buf_rsrc(W + (size_t)r0 * in, (uint32_t)(nrow * in));
  // every wave issues the same loads (wave 0's out of range: zeros, no
  // memory access), so the wait for x below counts exactly PC_LOADS later
  // loads on every path instead of draining them all
  uint4 w[PC_LOADS];
#pragma unroll
  for (int k = 0; k < PC_LOADS; ++k) {
    const int i = tid - 64 + 192 * k;
    w[k] = buf_load16(rw, wave > 0 && i < npiece ? (uint32_t)(i % PC_ROWS) * (uint32_t)in +
                                                       16u * (uint32_t)(i / PC_ROWS)
                                                 : 0xFFFFFFF0u);
  }
  if (tid < PC_LOADS) s_cnt[tid] = 0;
  if (tid < cblocks) ss[tid] = sv;
  __syncthreads();
#pragma unroll
  for (int q = 0; q < PC_XQ; ++q) {
    const int i = tid + 256 * q;
    if (i < in / 4) {
      float4 v = xv[q];
      if (MODE == 0) {  // xs = x * s of the row block (the 4 columns share a column block)
        const float sc = ss[(4 * i) / block];
        v = make_float4(v.x * sc, v.y * sc, v.z * sc, v.w * sc);
      }
      reinterpret_cast<float4 *>(xs)[i] = v;
    }
  }
  __syncthreads();
  if (wave > 0) {
#pragma unroll
    for (int k = 0; k < PC_LOADS; ++k) {
      const int i = tid - 64 + 192 * k;
      if (192 * k >= npiece) break;  // uniform
      if (i < npiece) pc_products<MODE>(w[k], i % PC_ROWS, 16 * (i / PC_ROWS), xs, ss, block, ps, pr);
      // this wave's product stores of load k are issued before the count (the
      // empty asm keeps the compiler from moving them past it; LDS runs a
      // wave's operations in order, so they land first): count the wave in
      asm volatile("" ::: "memory");
      if ((tid & 63) == 0) atomicAdd(&s_cnt[k], 1);
    }
    return;
  }
  if (tid >= PC_ROWS || tid >= nrow) return;
  const float4 *p4 = reinterpret_cast<const float4 *>(pr + (size_t)tid * ps);
  const int n4 = in / 4;  // a multiple of 8
  float acc = 0.0f;
  int ready = -1;  // loads known to be counted by all three producer waves
  auto wait_cols = [&](int cend) {  // products of columns < cend are in LDS
    const int need = (cend - 1) / 384;
    if (need <= ready) return;
    // (an LDS pointer: a generic one would make the read a FLAT one)
    const volatile __attribute__((address_space(3))) int *cnt =
        (const volatile __attribute__((address_space(3))) int *)&s_cnt[need];
    for (unsigned it = 0; *cnt < 3 && it < (1u << 24); ++it) __builtin_amdgcn_s_sleep(1);
    asm volatile("" ::: "memory");  // the product reads stay after the count's
    ready = need;
  };
  int b = 0;
#pragma unroll 1
  for (; b + 64 <= n4; b += 64) {
    wait_cols(4 * (b + 64));
    acc = pc_chain_fixed<64>(p4 + b, acc);
  }
  for (; b + 8 <= n4; b += 8) {
    wait_cols(4 * (b + 8));
    acc = pc_chain_fixed<8>(p4 + b, acc);
  }
  y[r0 + tid] = acc;
}

// The same product chains for longer rows, split (split chains,
// dsv4_device.h): the products do not depend on the sum, so a row is cut into
// 64 segments that run at once from guessed starts, and the serial part is a
// walk over groups of eight segments. A workgroup takes PS_ROWS rows, a wave
// per row, a lane per segment with all 8 candidates in registers. Thread t
// forms the products of columns 16 t .. + 15 of every row (its x and scale
// stay in registers) and their sum in double; lane s then chooses the start of
// segment s among the middle six multiples of 8 columns of its 64 by the
// largest |prefix| (by simulation 0.2 segments of a row miss, 3.6 without). The candidates stay within 20 grid steps of the start of each
// other (7 at the start; a tie may add one step per grid, a coarser grid its
// own step, at most two binades up), so the margin of the first one less 32
// steps serves them all. Bound: instruction issue of the candidates' chains
// (12 per column and segment, on segments as long as the longest of the wave's,
// about 1.7 times the mean), then the serial walk and the first memory round
// trip; 2048 x 4096: 15.0 us, 21.0 us as one add chain per row; 50 us where every
// segment misses (each pair of products all but cancelling).
#define PS_ROWS 4
#define PS_MININ 1024
#define PS_MAXIN 4096  // 64 segments of 64 columns
#define PS_REC 10  // dwords per record: r[8], base | binades up, margin
__host__ __device__ constexpr int ps_pr(int in) { return PS_ROWS * (sp_at(in - 16) + 16); }
// the products, then the sums of the 16-column chunks (double) and of their
// first halves (float), whose place the records take
static size_t ps_lds(int in) { return ((size_t)ps_pr(in) + PS_ROWS * 256 * 3) * 4; }

// acc + the products of columns [c, e), in order (c, e multiples of 8); the
// next 8 are read while 8 are added.
__device__ __forceinline__ float ps_chain(const float *p, int c, int e, float acc) {
  const float4 *q = reinterpret_cast<const float4 *>(p + sp_at(c));
  float4 v0 = q[0], v1 = q[1];
  for (; c < e; c += 8) {
    q = reinterpret_cast<const float4 *>(p + sp_at(min(c + 8, e - 8)));
    const float4 n0 = q[0], n1 = q[1];
    acc = acc + v0.x;
    acc = acc + v0.y;
    acc = acc + v0.z;
    acc = acc + v0.w;
    acc = acc + v1.x;
    acc = acc + v1.y;
    acc = acc + v1.z;
    acc = acc + v1.w;
    v0 = n0;
    v1 = n1;
  }
  return acc;
}

template <int MODE>
__global__ __launch_bounds__(64 * PS_ROWS) void k_fp8_prodsplit(float *__restrict__ y,
                                                                const float *__restrict__ x,
                                                                const uint8_t *__restrict__ W,
                                                                const float *__restrict__ wscale,
                                                                int in, int rows, int block) {
  extern __shared__ __align__(16) float lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int row = __builtin_amdgcn_readfirstlane(tid >> 6), r0 = blockIdx.x * PS_ROWS;
  const int cblocks = (in + block - 1) / block, nch = in / 16;
  const int rs = ps_pr(in) / PS_ROWS;  // product row stride
  float *rec = lds + ps_pr(in) + row * 64 * PS_REC;
  double *ps = reinterpret_cast<double *>(lds + ps_pr(in));  // [PS_ROWS][256], before rec
  float *ph = reinterpret_cast<float *>(ps + PS_ROWS * 256);  // [PS_ROWS][256]
  if (tid < nch) {
    float4 xv[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) xv[q] = reinterpret_cast<const float4 *>(x)[4 * tid + q];
    const float sc = wscale[(size_t)(r0 / block) * cblocks + 16 * tid / block];
    const BufRsrc rw = buf_rsrc(W + (size_t)r0 * in, (uint32_t)(min(PS_ROWS, rows - r0) * in));
    uint4 w[PS_ROWS];
#pragma unroll
    for (int r = 0; r < PS_ROWS; ++r) w[r] = buf_load16(rw, (uint32_t)(r * in + 16 * tid));
    if (MODE == 0)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        xv[q] = make_float4(xv[q].x * sc, xv[q].y * sc, xv[q].z * sc, xv[q].w * sc);
#pragma unroll
    for (int r = 0; r < PS_ROWS; ++r) {
      const uint32_t wd[4] = {w[r].x, w[r].y, w[r].z, w[r].w};
      double sum = 0.0;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        if (d == 2) ph[r * 256 + tid] = (float)sum;
        const float2 lo = fp8x2<false>(wd[d]), hi = fp8x2<true>(wd[d]);
        float4 p = make_float4(lo.x * xv[d].x, lo.y * xv[d].y, hi.x * xv[d].z, hi.y * xv[d].w);
        if (MODE == 1) p = make_float4(p.x * sc, p.y * sc, p.z * sc, p.w * sc);
        *reinterpret_cast<float4 *>(lds + r * rs + sp_at(16 * tid) + 4 * d) = p;
        sum += ((double)p.x + (double)p.y) + ((double)p.z + (double)p.w);
      }
      ps[r * 256 + tid] = sum;
    }
  }
  __syncthreads();
  // ---- lane s: prefixes of its 4 chunks, its segment's start and guess
  const int nseg = (nch + 3) / 4;
  int beg = 0;
  uint32_t base = 0;
  {
    double v[4], tot = 0.0;
    float half[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int at = row * 256 + min(4 * lane + q, nch - 1);
      v[q] = 4 * lane + q < nch ? ps[at] : 0.0;
      half[q] = ph[at];
      tot += v[q];
    }
    double inc = tot;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const double u = __shfl_up(inc, o);
      if (lane >= o) inc += u;
    }
    double pre = inc - tot;
    float best = -1.0f;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const float g = (float)(q % 2 ? pre + (double)half[q / 2] : pre);
      if (q > 0 && q < 7 && 4 * lane + q / 2 < nch && fabsf(g) > best) {
        best = fabsf(g);
        beg = 64 * lane + 8 * q;
        base = f2u(g) & ~7u;
      }
      if (q % 2) pre += v[q / 2];
    }
    if (lane == 0 || best < 0.0f) {  // the chain's own start; NaN prefixes
      beg = 64 * lane;
      base = 0;
    }
  }
  const int nxt = __shfl_down(beg, 1), end = lane + 1 < nseg ? nxt : in;
  __syncthreads();  // ps is read; rec takes its place
  // ---- the segments
  float mgn = __builtin_inff(), top = 0.0f, r[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = u2f(base | j);
  const float *pr = lds + row * rs;
  if (lane < nseg) {
    const float4 *q4 = reinterpret_cast<const float4 *>(pr + sp_at(beg));
    float4 v[2] = {q4[0], q4[1]};
    for (int c = beg; c < end; c += 8) {
      q4 = reinterpret_cast<const float4 *>(pr + sp_at(min(c + 8, end - 8)));
      const float4 n[2] = {q4[0], q4[1]};
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const float pv[4] = {v[q].x, v[q].y, v[q].z, v[q].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
          for (int j = 0; j < 8; ++j) r[j] = r[j] + pv[i];
          // the smaller distance to the binade's ends b, 2 b: b / 2 less that
          // to its middle (each step exact)
          const float b = u2f(f2u(r[0]) & 0xFF800000u), mid = fmaf(-1.5f, b, r[0]);
          mgn = fminf(mgn, fmaf(0.5f, fabsf(b), -fabsf(mid)));
          top = fmaxf(top, fabsf(r[0]));
        }
      }
      v[0] = n[0];
      v[1] = n[1];
    }
    // binades up; an infinite result (its distances are NaN, which the minimum
    // drops) allows no shift
    const int te = (int)(f2u(top) >> 23);
    const int up = te < 255 ? te - (int)((base >> 23) & 255u) : 7;
    // 32 grid steps of the start: its last place times 32
    const float step = fabsf(u2f(base | 1u) - u2f(base));
    const float m = up <= 2 ? mgn * 0.999f - 32.0f * step : 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) rec[lane * PS_REC + j] = r[j];
    rec[lane * PS_REC + 8] = u2f(base | (uint32_t)max(0, min(up, 7)));
    rec[lane * PS_REC + 9] = m > 0.0f ? m : 0.0f;
  }
  __syncthreads();
  // ---- eight segments at a time: lane = (group lane / 8, candidate lane % 8)
  const int ngrp = (nseg + 7) / 8, s0 = 8 * (lane >> 3);
  float gend = 0.0f, gm = -1.0f;
  uint32_t gbase = 0;
  if (s0 < nseg) {
    gbase = f2u(rec[s0 * PS_REC + 8]) & ~7u;
    float a = u2f(gbase | (lane & 7)), m = __builtin_inff();
    int up = 0;
    bool ok = true;
    for (int s = s0; s < min(s0 + 8, nseg); ++s) {
      const float *R = rec + s * PS_REC;
      const uint32_t b = f2u(R[8]);
      float e, left;
      ok = sp_step(a, b & ~7u, R[f2u(a) & 7], R[9], &e, &left) && ok;
      up = max(up, (int)(b >> 23 & 255u) + (int)(b & 7u));
      a = e;
      m = fminf(m, left);
    }
    gend = a;
    gm = !ok ? -1.0f : up <= (int)(gbase >> 23 & 255u) + 2 && m > 0.0f ? m : 0.0f;
  }
  // ---- the walk (every lane the same)
  float a = 0.0f;
  for (int q = 0; q < ngrp; ++q) {
    const int j = __builtin_amdgcn_readfirstlane((int)(f2u(a) & 7u)) + 8 * q;
    const uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)gbase, 8 * q);
    const float m = u2f(__builtin_amdgcn_readlane(f2u(gm), j));
    float e, left;
    if (sp_step(a, b, u2f(__builtin_amdgcn_readlane(f2u(gend), j)), m, &e, &left) && m >= 0.0f) {
      a = e;
      continue;
    }
    for (int s = 8 * q; s < min(8 * q + 8, nseg); ++s) {
      const float *R = rec + s * PS_REC;
      if (sp_step(a, f2u(R[8]) & ~7u, R[f2u(a) & 7], R[9], &e, &left))
        a = e;
      else
        a = ps_chain(pr, __builtin_amdgcn_readlane(beg, s), __builtin_amdgcn_readlane(end, s), a);
    }
  }
  if (lane == 0 && r0 + row < rows) y[r0 + row] = a;
}

// ================================================ batched BF16 rows ====
// dsv4_gemv_bf16_batch / head_logits_batch (src/dsv4/dsv4_model.c:266-367,
// 7371-7445) for 1 to 64 tokens on the fp32 matrix unit. v_mfma_f32_16x16x4
// adds its four products to the accumulator one after another in k order,
// each as one rounded fma with subnormals kept (test_f32_mfma_is_fma_chain
// checks the bits), so a tile fed four columns at a time runs the reference's
// column-order fmaf chain of each (row, token). Bound: the fp32 matrix rate,
// 256 FLOP per clock and CU, twice the VALU's (64 tokens through the 129280 x
// 4096 head are 34 G fma: 437 us at that rate, 540 us here, 1000 us as VALU chains; 16 tokens are
// HBM-bound, 220 us against 700). Smaller matrices, whose VALU chains left
// waves waiting, gain most: 16384 rows, 64 tokens 654 -> 90 us.
//
// A workgroup of 4 waves takes 64 MR rows, a wave 16 MR rows x 16 NT tokens
// (MR NT accumulator tiles: independent chains hide an MFMA's latency, 33
// clocks back to back on one tile, 50 with an operand formed in between). Per
// step of 64 columns a wave loads its rows coalesced (8 lanes per 128-byte
// piece, D steps in flight) and writes them to its own LDS rows: one row tile
// (WIDE) widened and split by c % 4, so that one 16-byte read is a lane's
// operand of four MFMAs and nothing stands between them (router of 777 tokens
// 63 -> 47 us); more row tiles as they are (144 bytes apart: conflict-free),
// read back per (row, 8 columns), v_perm widening the lane's column of each
// four, which the other tiles' MFMAs cover. x is staged once per workgroup,
// split by c % 4 as well, double-buffered. The x
// loads of a step are issued ahead of its weights (loads complete in order).
//
// ROUTER: the gate's rows; y is the scores sqrt(softplus(z)), choice the
// scores plus the bias, and blockIdx.y the token tile.
// LDS floats per token of an x tile: 64 + 4. (Rows of 80 floats with rotated
// chunks, mt_at, write without conflicts, but leave fewer workgroups per CU: 80000
// rows, 64 tokens 347 -> 427 us.)
#define RM_XS 68
template <int NT, int MR, bool ROUTER>
__global__ __launch_bounds__(256, 2) void k_bf16_rows_mfma(float *__restrict__ y,
                                                           const float *__restrict__ x,
                                                           const uint16_t *__restrict__ W,
                                                           int in, int rows, int round_out,
                                                           int t0, int nt, float *__restrict__ choice,
                                                           const float *__restrict__ bias) {
  if (ROUTER) {
    t0 = blockIdx.y * 16 * NT;
    nt = min(16 * NT, nt - t0);
  }
  constexpr int D = NT * MR <= 2 ? 4 : 2;  // steps in flight
  __shared__ __align__(16) float xs[2][16 * NT * RM_XS];
  constexpr bool WIDE = MR == 1;
  __shared__ __align__(16) uint4 tl[4][16 * MR * (WIDE ? RM_XS / 4 : 9)];
  constexpr int LD = 2 * MR;  // 16-byte weight loads per lane and step
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  const int r0 = (blockIdx.x * 4 + wave) * 16 * MR;
  const int nrow = __builtin_amdgcn_readfirstlane(max(0, min(16 * MR, rows - r0)));
  const uint32_t rb = 2u * (uint32_t)in;
  const BufRsrc rw = buf_rsrc(W + (size_t)r0 * in, (uint32_t)nrow * rb);
  const BufRsrc rx = buf_rsrc(x + (size_t)t0 * in, (uint32_t)nt * 2u * rb);
  const int lr = lane >> 3, lp = lane & 7;
  const uint32_t lo = (uint32_t)lr * rb + 16u * lp;  // step t, rows 8 i + lr: + 8 rb i + 128 t
  const int steps = in / 64;
  // x staging: thread = (token tid / 4, 16 columns 16 (tid % 4) of the step);
  // every load is issued without a branch, past the last step or token out of
  // range (zeros, no access); tokens past the run are not stored
  const uint32_t xo = (uint32_t)(tid >> 2) * 2u * rb + 64u * (uint32_t)(tid & 3);
  const int xd = (tid >> 2) * RM_XS + 4 * (tid & 3);
  // bytes of the lane's column of four (two dwords) as a widened BF16
  const uint32_t sel = 0x01000C0Cu + 0x02020000u * (uint32_t)g;
  uint4 xr[D][4], T[D][LD];
  auto load = [&](int d, int t) {
    const uint32_t xn = t < steps ? xo + 256u * (uint32_t)t : 0xFFFFFF00u;
#pragma unroll
    for (int j = 0; j < 4; ++j) xr[d][j] = buf_load16(rx, xn + 16u * j);
#pragma unroll
    for (int i = 0; i < LD; ++i)
      T[d][i] = buf_load16(rw, t < steps ? lo + 8u * rb * i + 128u * t : 0xFFFFFFF0u);
  };
#pragma unroll
  for (int d = 0; d < D; ++d) load(d, d);
  f32x4 acc[MR][NT];
#pragma unroll
  for (int m = 0; m < MR; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int tb = 0; tb < steps; tb += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int t = tb + d;
      float *xw = xs[d % 2];
      if (64 * NT == 256 || tid < 64 * NT) {
        const uint4 *c = xr[d];
        *reinterpret_cast<uint4 *>(xw + xd) = make_uint4(c[0].x, c[1].x, c[2].x, c[3].x);
        *reinterpret_cast<uint4 *>(xw + xd + 16) = make_uint4(c[0].y, c[1].y, c[2].y, c[3].y);
        *reinterpret_cast<uint4 *>(xw + xd + 32) = make_uint4(c[0].z, c[1].z, c[2].z, c[3].z);
        *reinterpret_cast<uint4 *>(xw + xd + 48) = make_uint4(c[0].w, c[1].w, c[2].w, c[3].w);
      }
#pragma unroll
      for (int i = 0; i < LD; ++i) {
        const uint4 v = T[d][i];
        if (WIDE) {
          float2 *wd = reinterpret_cast<float2 *>(tl[wave]) + (8 * i + lr) * (RM_XS / 2) + lp;
          wd[0] = make_float2(u2f(v.x << 16), u2f(v.z << 16));
          wd[8] = make_float2(u2f(v.x & 0xFFFF0000u), u2f(v.z & 0xFFFF0000u));
          wd[16] = make_float2(u2f(v.y << 16), u2f(v.w << 16));
          wd[24] = make_float2(u2f(v.y & 0xFFFF0000u), u2f(v.w & 0xFFFF0000u));
        } else {
          tl[wave][(8 * i + lr) * 9 + lp] = v;
        }
      }
      load(d, t + D);
      __syncthreads();
      if (t >= steps) break;  // uniform; the last round may be short
      // eight pieces of 8 columns: the reads of a piece are issued ahead of the
      // MFMAs of the one before it (the empty asm keeps the compiler from
      // hoisting every read of the step, which spilled)
      f32x4 b[2][NT];
      uint4 w[2][MR];
      auto read = [&](int p) {
        if (p % 2 == 0)
#pragma unroll
          for (int n = 0; n < NT; ++n)
            b[p / 2 % 2][n] =
                *reinterpret_cast<const f32x4 *>(xw + (16 * n + l16) * RM_XS + 16 * g + 2 * p);
#pragma unroll
        for (int m = 0; m < MR; ++m) {
          if (!WIDE)
            w[p % 2][m] = tl[wave][(16 * m + l16) * 9 + p];
          else if (p % 2 == 0)
            w[p / 2 % 2][m] = tl[wave][(16 * m + l16) * (RM_XS / 4) + 4 * g + p / 2];
        }
      };
      read(0);
#pragma unroll
      for (int p = 0; p < 8; ++p) {
        asm volatile("" ::: "memory");
        if (p + 1 < 8) read(p + 1);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 2; ++e)  // 4 columns
#pragma unroll
          for (int m = 0; m < MR; ++m) {
            const uint4 wm = w[WIDE ? p / 2 % 2 : p % 2][m];
            const float av = u2f(WIDE ? p % 2 ? e ? wm.w : wm.z : e ? wm.y : wm.x
                                 : e  ? __builtin_amdgcn_perm(wm.w, wm.z, sel)
                                      : __builtin_amdgcn_perm(wm.y, wm.x, sel));
#pragma unroll
            for (int n = 0; n < NT; ++n)
              acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                  av, b[p / 2 % 2][n][2 * (p % 2) + e], acc[m][n], 0, 0, 0);
          }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int tok = 16 * n + l16;
    if (tok >= nt) continue;
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = 16 * m + 4 * g + v;
        const float o = acc[m][n][v];
        const size_t at = (size_t)(t0 + tok) * rows + r0 + row;
        if (row < nrow) {
          if (ROUTER) {
            const float sc = sqrt_softplus(o);
            y[at] = sc;
            choice[at] = sc + (bias ? bias[r0 + row] : 0.0f);
          } else {
            y[at] = round_out ? bf16_round(o) : o;
          }
        }
      }
  }
}

// The same chains for a few tokens of many or narrow rows (tiled_width), where HBM
// or the launch is the bound: a lane per output row reading its own row would touch 64 cache lines per load,
// so the wave loads tiles of 64 rows x 64 columns coalesced (lane l: rows
// 8 i + l / 8, 16 bytes at column 8 (l % 8)), writes them to LDS (rows 144
// bytes apart, so that the lanes' row reads hit distinct banks) and reads back
// its own row's 64 columns. Two tiles are in flight while one is chained; x
// enters each fmaf as a scalar operand. LDS holds one tile: the wave's LDS
// accesses run in order, and the empty asms keep the compiler from moving them
// across each other. in a multiple of 64; tokens [t0, t0 + TB) present. 129280 x
// 4096: 180 to 187 us, and 220 where the matrix lies badly in memory (one
// allocation in ten, the same each time it is read); 2 tokens 206.
#define RT_DEPTH 2
template <int TB>
__global__ __launch_bounds__(64) void k_bf16_rows_tiled(float *__restrict__ y,
                                                        const float *__restrict__ x,
                                                        const uint16_t *__restrict__ W, int in,
                                                        int rows, int round_out, int t0) {
  __shared__ __align__(16) uint4 tl[64 * 9];
  const int lane = threadIdx.x, r0 = blockIdx.x * 64;
  const int nrow = min(64, rows - r0);
  const uint32_t rb = 2u * (uint32_t)in;
  const BufRsrc rw = buf_rsrc(W + (size_t)r0 * in, (uint32_t)nrow * rb);
  const int lr = lane >> 3, lp = lane & 7;
  const uint32_t lo = (uint32_t)lr * rb + 16u * lp;  // tile t, rows 8 i + lr: + 8 rb i + 128 t
  const int nt = in / 64;
  typedef const __attribute__((address_space(4))) float cfloat;
  cfloat *xc = (cfloat *)(x + (size_t)t0 * in);
  uint4 T[RT_DEPTH][8];
#pragma unroll
  for (int d = 0; d < RT_DEPTH; ++d)
#pragma unroll
    for (int i = 0; i < 8; ++i)
      T[d][i] = buf_load16(rw, d < nt ? lo + 8u * rb * i + 128u * d : 0xFFFFFFF0u);
  float acc[TB];
#pragma unroll
  for (int t = 0; t < TB; ++t) acc[t] = 0.0f;
  for (int tb = 0; tb < nt; tb += RT_DEPTH) {
#pragma unroll
    for (int d = 0; d < RT_DEPTH; ++d) {
      const int t = tb + d;
      if (t >= nt) break;  // uniform
      asm volatile("" ::: "memory");
#pragma unroll
      for (int i = 0; i < 8; ++i) tl[(8 * i + lr) * 9 + lp] = T[d][i];
      if (t + RT_DEPTH < nt) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          T[d][i] = buf_load16(rw, lo + 8u * rb * i + 128u * (t + RT_DEPTH));
      }
      asm volatile("" ::: "memory");
      uint4 m[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) m[k] = tl[lane * 9 + k];
      asm volatile("" ::: "memory");
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t wd[4] = {m[k].x, m[k].y, m[k].z, m[k].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int c = 64 * t + 8 * k + 2 * e;
          const float wl = u2f(wd[e] << 16), wh = u2f(wd[e] & 0xFFFF0000u);
#pragma unroll
          for (int u = 0; u < TB; ++u) {
            acc[u] = fmaf(wl, xc[(size_t)u * in + c], acc[u]);
            acc[u] = fmaf(wh, xc[(size_t)u * in + c + 1], acc[u]);
          }
        }
      }
    }
  }
  if (lane >= nrow) return;
#pragma unroll
  for (int u = 0; u < TB; ++u)
    y[(size_t)(t0 + u) * rows + r0 + lane] = round_out ? bf16_round(acc[u]) : acc[u];
}

// ======================================================= greedy pick ===
// The CLI's greedy token (src/cli/dsv4_run.c:357-359): best = 0, then every
// v with logits[v] > logits[best] in order; so the first index of the
// largest value, NaNs never taken, and 0 when logits[0] is NaN. One
// workgroup per row. Bound: one CU's load rate and latency (517 KB per row
// at the model's vocabulary), so 16 waves with 8 16-byte loads each in
// flight: 147 us with 4 waves and one 4-byte load in flight each, about 8 us
// now (one row of 129280); fewer waves and loads for shorter rows
// (dsv4g_argmax). A thread's loads past the row are clamped to
// the row's last 4 values (seen twice, which changes nothing). Each thread
// keeps the first largest value of its ascending indices (bi < 0: none above
// -inf; a row with no value above -inf gives 0, as the rule does whether
// logits[0] is -inf or NaN), then (value, index) pairs merge with the larger
// value, or the smaller index on equal values.
__device__ __forceinline__ void am_merge(float &bv, int &bi, float ov, int oi) {
  if (oi >= 0 && (bi < 0 || ov > bv || (ov == bv && oi < bi))) {
    bv = ov;
    bi = oi;
  }
}

// T threads per row, Q 16-byte loads in flight per thread.
template <int AM_T, int AM_Q>
__global__ __launch_bounds__(AM_T) void k_argmax(int *idx, const float *logits, int vocab,
                                                 size_t stride) {
  __shared__ float s_v[AM_T / 64];
  __shared__ int s_i[AM_T / 64];
  const int tid = threadIdx.x;
  const float *l = logits + (size_t)blockIdx.x * stride;
  float bv = -__builtin_inff();
  int bi = -1;
  auto take = [&](float f, int i) {  // false for NaN
    const bool t = f > bv;
    bv = t ? f : bv;
    bi = t ? i : bi;
  };
  if (vocab >= 4) {
    for (long b = 0; b < vocab; b += 4 * AM_T * AM_Q) {
      float4 f[AM_Q];
      int at[AM_Q];
#pragma unroll
      for (int k = 0; k < AM_Q; ++k) {
        at[k] = (int)min(b + 4 * (tid + AM_T * k), (long)vocab - 4);
        __builtin_memcpy(&f[k], l + at[k], 16);  // rows may start at any float
      }
#pragma unroll
      for (int k = 0; k < AM_Q; ++k) {
        take(f[k].x, at[k]);
        take(f[k].y, at[k] + 1);
        take(f[k].z, at[k] + 2);
        take(f[k].w, at[k] + 3);
      }
    }
  } else if (tid < vocab) {
    take(l[tid], tid);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
    am_merge(bv, bi, __shfl_xor(bv, o, 64), __shfl_xor(bi, o, 64));
  if (tid % 64 == 0) {
    s_v[tid / 64] = bv;
    s_i[tid / 64] = bi;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < AM_T / 64; ++w) am_merge(bv, bi, s_v[w], s_i[w]);
    const float f0 = l[0];
    idx[blockIdx.x] = (f0 != f0 || bi < 0) ? 0 : bi;
  }
}

// ============================================= public float-scale GEMVs ===
// dsv4_gemv_fp8 / dsv4_gemv_fp8_tbl (src/dsv4/dsv4_ops.c:176-239) and
// dsv4_gemv_fp4 (src/dsv4/dsv4_ops.c:249-284): one sequential chain per row,
// unfused (the reference builds with -ffp-contract=off), here one lane per
// row with the same expression and column order. Bit-exact.
// mode 0 (dsv4_gemv_fp8): acc += w * (x * s); mode 1 (_tbl): acc += (w * x) * s.
__global__ __launch_bounds__(64) void k_gemv_fp8_float(float *__restrict__ y,
                                                       const float *__restrict__ x,
                                                       const uint8_t *__restrict__ W,
                                                       const float *__restrict__ wscale, int in,
                                                       int rows, int block, int mode) {
  const int row = blockIdx.x * 64 + threadIdx.x;
  if (row >= rows) return;
  const int cblocks = (in + block - 1) / block;
  const float *srow = wscale + (size_t)(row / block) * cblocks;
  const uint8_t *wr = W + (size_t)row * in;
  float acc = 0.0f;
  for (int c = 0; c < in; ++c) {
    const float w = e4m3_decode(wr[c]);
    const float s = srow[c / block];
    acc += mode == 0 ? w * (x[c] * s) : (w * x[c]) * s;
  }
  y[row] = acc;
}

// acc += (w * (qx * qs)) * ws, columns in order
__global__ __launch_bounds__(64) void k_gemv_fp4_float(float *__restrict__ y,
                                                       const float *__restrict__ qx,
                                                       const float *__restrict__ qscale,
                                                       const uint8_t *__restrict__ W,
                                                       const float *__restrict__ wscale, int in,
                                                       int rows, int group) {
  const int row = blockIdx.x * 64 + threadIdx.x;
  if (row >= rows) return;
  const size_t pcols = (size_t)(in + 1) / 2, gcols = (size_t)(in + group - 1) / group;
  const uint8_t *wr = W + (size_t)row * pcols;
  const float *ws = wscale + (size_t)row * gcols;
  float acc = 0.0f;
  for (int c = 0; c < in; ++c) {
    const uint32_t b = wr[c >> 1];
    const float w = e2m1_decode((c & 1) ? (b >> 4) : (b & 15u));
    const float xd = qx[c] * qscale[c / 128];
    acc += (w * xd) * ws[c / group];
  }
  y[row] = acc;
}

// ================================================ synthetic quantisers ===
// Build checkpoints in the reference formats from fp32 weights. The rules
// are the reference's activation rules applied to weights: E8M0 scale
// 2^ceil(log2(amax/6)) per 32 (FP4, nearest E2M1 with ties to the even code,
// src/dsv4/dsv4_model.c:1420-1447) or 2^ceil(log2(amax/448)) per 128x128
// block (FP8), or the fp32 absmax/448 block scale of the public FP8 GEMV.
__device__ __forceinline__ uint32_t fp4_code(float q) {
  const float mag[8] = {0.0f, 0.5f, 1.0f, 1.5f, 2.0f, 3.0f, 4.0f, 6.0f};
  const float a = fabsf(q);
  int best = 0;
  float bd = a;
  for (int k = 0; k < 8; ++k) {
    const float d = fabsf(a - mag[k]);
    if (d < bd) {
      bd = d;
      best = k;
    } else if (d == bd && (k & 1) == 0) {
      best = k;
    }
  }
  return (uint32_t)best | (q < 0.0f ? 8u : 0u);
}

__device__ __forceinline__ int pow2_ceil_exp(float r) {
  int e;
  const float m = frexpf(r, &e);
  if (m == 0.5f) e--;
  return e;
}

// One thread per (row, 32-group).
__global__ void k_quant_fp4_rows(uint8_t *__restrict__ packed, uint8_t *__restrict__ scales,
                                 const float *__restrict__ w, int rows, int cols) {
  const int gcols = cols / 32;
  const size_t idx = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (idx >= (size_t)rows * gcols) return;
  const size_t r = idx / gcols, g = idx % gcols;
  const float *wr = w + r * cols + g * 32;
  float amax = 0.0f;
  for (int i = 0; i < 32; ++i) amax = fmaxf(amax, fabsf(wr[i]));
  const float floor_amax = 6.0f * 0x1p-126f;
  if (amax < floor_amax) amax = floor_amax;
  const int e = pow2_ceil_exp(amax * (1.0f / 6.0f));
  scales[idx] = (uint8_t)(e + 127);
  const float inv = 1.0f / ldexpf(1.0f, e);
  uint8_t *pr = packed + r * (cols / 2) + g * 16;
  for (int i = 0; i < 16; ++i) {
    float q0 = wr[2 * i] * inv, q1 = wr[2 * i + 1] * inv;
    q0 = fminf(fmaxf(q0, -6.0f), 6.0f);
    q1 = fminf(fmaxf(q1, -6.0f), 6.0f);
    pr[i] = (uint8_t)(fp4_code(q0) | (fp4_code(q1) << 4));
  }
}

// One workgroup per 128x128 block. mode 0: E8M0 scale codes (uint8);
// mode 1: fp32 absmax/448 scales.
__global__ __launch_bounds__(256) void k_quant_fp8_blocks(uint8_t *__restrict__ codes,
                                                          void *__restrict__ scales,
                                                          const float *__restrict__ w,
                                                          int rows, int cols, int mode) {
  __shared__ float red[4];
  const int cb = (cols + 127) / 128;
  const int br = blockIdx.x / cb, bc = blockIdx.x % cb;
  const int r0 = br * 128, c0 = bc * 128;
  const int r1 = min(r0 + 128, rows), c1 = min(c0 + 128, cols);
  float amax = 0.0f;
  for (int i = threadIdx.x; i < 128 * 128; i += 256) {
    const int r = r0 + i / 128, c = c0 + i % 128;
    if (r < r1 && c < c1) amax = fmaxf(amax, fabsf(w[(size_t)r * cols + c]));
  }
  amax = wave_max(amax);
  if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float inv;
  bool divide = false;
  float s = 1.0f;
  if (mode == 0) {
    const float a = amax < 1e-4f ? 1e-4f : amax;
    const int e = pow2_ceil_exp(a * (1.0f / 448.0f));
    if (threadIdx.x == 0) reinterpret_cast<uint8_t *>(scales)[blockIdx.x] = (uint8_t)(e + 127);
    inv = 1.0f / ldexpf(1.0f, e);
  } else {
    s = amax > 0.0f ? amax / 448.0f : 1.0f;
    if (threadIdx.x == 0) reinterpret_cast<float *>(scales)[blockIdx.x] = s;
    inv = 0.0f;
    divide = true;
  }
  for (int i = threadIdx.x; i < 128 * 128; i += 256) {
    const int r = r0 + i / 128, c = c0 + i % 128;
    if (r < r1 && c < c1) {
      const float v = w[(size_t)r * cols + c];
      float q = divide ? v / s : v * inv;
      if (q > 448.0f) q = 448.0f;
      else if (q < -448.0f) q = -448.0f;
      codes[(size_t)r * cols + c] = (uint8_t)e4m3_code(round_e4m3(q));
    }
  }
}

}  // namespace dsv4

// ============================================================ C-ABI =====
using namespace dsv4;

template <int NP>
static void launch_fp4_t(const GemvArgs *a, int nvec, int pair, hipStream_t st) {
  const Fp4Geom q = fp4_geom_np(a->in, NP);
  const int span = pair ? q.tr / 2 : q.tr;
  const dim3 grid((unsigned)((a->rows + span - 1) / span), (unsigned)nvec);
  const size_t lds = (size_t)q.tr * pair_stride(q.G) * 8 + 4096 + ((a->in + 15) & ~15) +
                     (size_t)((a->in + 127) / 128) * 4;
  hipLaunchKernelGGL(k_gemv_fp4_t<NP>, grid, dim3(256), lds, st, *a, pair);
}

// Row tiles per wave: 4 up to 16 tokens, else 2, where that leaves the busiest
// CU no more tiles than one each (workgroups per CU times tiles) and every CU
// more than one workgroup, so that one computes while another stages; else 1.
// Rows of 4096 columns, us with 1 / 4 tiles at 16 tokens: 65536 rows 129 / 145,
// 98304 185 / 204, 114688 217 / 208, 120000 235 / 212, 129280 245 / 222, 150000
// 302 / 333; with 1 / 2 at 64 tokens: 57344 348 / 279, 65536 359 / 280, 73728 361 /
// 392, 90112 431 / 394, 114688 536 / 538, 129280 572 / 543. (2 at 16 tokens and 4
// beyond gave nothing: 256 and 547 at 129280.) Rows of up to 128 columns are
// mostly a workgroup's start: the larger tile up to 32 tokens as soon as it fills
// the CUs (100000 x 64, 16 tokens 13.1 / 10.4, 32 tokens 18.4 / 16.8).
template <int NT>
static void launch_rows_mfma_nt(float *y, const float *x, const uint16_t *W, int in, int out,
                                int round_out, int t0, int n, hipStream_t st) {
  constexpr int MR = NT == 1 ? 4 : 2;
  const long one = (out + 63L) / 64, wgs = (out + 64L * MR - 1) / (64L * MR);
  const bool tiles = wgs > 256 && ((wgs + 255) / 256 * MR <= (one + 255) / 256 ||
                                   (NT <= 2 && in <= 128));
  auto k = tiles ? k_bf16_rows_mfma<NT, MR, false> : k_bf16_rows_mfma<NT, 1, false>;
  hipLaunchKernelGGL(k, dim3((unsigned)(tiles ? wgs : one)), dim3(256), 0, st, y, x, W, in, out,
                     round_out, t0, n, nullptr, nullptr);
}

static void launch_rows_mfma(float *y, const float *x, const uint16_t *W, int in, int out,
                             int round_out, int t0, int n, hipStream_t st) {
  if (n <= 16)
    launch_rows_mfma_nt<1>(y, x, W, in, out, round_out, t0, n, st);
  else if (n <= 32)
    launch_rows_mfma_nt<2>(y, x, W, in, out, round_out, t0, n, st);
  else if (n <= 48)
    launch_rows_mfma_nt<3>(y, x, W, in, out, round_out, t0, n, st);
  else
    launch_rows_mfma_nt<4>(y, x, W, in, out, round_out, t0, n, st);
}

// The widest rows that n tokens take through the tiled chains. Those wait on
// memory and their own latency, about the same time however many waves a CU has,
// and issue an fma per token and column; the matrix unit's wait less and cost as
// much for one token as for 16, once per workgroup of 64 rows, so many rows (w =
// 64-row tiles per CU) favour the tiled form and wide rows or more tokens the
// matrix unit's (us, tiled / matrix unit). One token: 16384 rows of 128 3.5 / 4.0,
// of 256 5.3 / 4.7; 40000 of 384 10.0 / 11.5, of 512 15.7 / 13.6; 72000 of 512
// 20.1 / 21.4, of 4096 163 / 147; 98304 of 1024 40 / 44, of 4096 185 / 166; 106496
// of 4096 185 / 194; 129280 180 / 210. Two: 24000 of 192 5.4 / 6.2, of 256 6.7 /
// 6.6; 96000 of 512 23.8 / 25.2, of 1024 45.2 / 44.2; 100000 of 1024 45.6 / 50.7, of
// 4096 198 / 195; 129280 of 4096 206 / 210. Three:
// 50000 of 256 8.9 / 10.3; 100000 of 768 38.8 / 39.6, of 1024 53 / 51. Four:
// 65536 of 192 7.5 / 10, of 256 12.0 / 11.0. Eight: 65536 of 64 4.7 / 7.1, of 128
// 9.0 / 8.6; 100000 of 128 10.0 / 13.1, of 192 15.9 / 15.9. (16 tokens
// through 100000 x 64 took 8.8 and 32 13.7 with four rows a lane on the VALU,
// here 10.4 and 16.8; that form lost everywhere else and is gone.)
static int tiled_width(int n, int out) {
  constexpr int ANY = 0x7fffffff;
  //                             w = 1    2    3    4    5    6     7   more
  static constexpr int W[5][8] = {{128, 384, 384, 384, 512, 1024, ANY, ANY},  // 1 token
                                  {64, 192, 320, 320, 384, 512, 1024, ANY},   // 2
                                  {64, 128, 192, 256, 256, 384, 768, 768},    // 3
                                  {64, 64, 192, 192, 192, 192, 384, 384},     // 4
                                  {0, 64, 64, 64, 128, 128, 128, 128}};       // 8
  if (n > 4 && n != 8) return 0;
  return W[n == 8 ? 4 : n - 1][std::min((out + 16383L) / 16384, 8L) - 1];
}

// Every (token, expert) score and choice of the batched router, [T][E], exact.
// Token tiles per wave: the fewest with at most one workgroup per CU (256
// experts, beside the shared expert's GEMMs: 53 us at 300 tokens, 61 at 777, 92 at
// 2048, 143 at 3400; 44, 54, 80 and 121 at the least).
int dsv4g_launch_router_scores(float *score, float *choice, const float *x, const uint16_t *G,
                               const float *bias, int T, int H, int E, hipStream_t st) {
  const int egroups = (E + 63) / 64;
  const long tiles = (T + 15L) / 16 * egroups;
  const int nt = tiles <= 256 ? 1 : tiles <= 512 ? 2 : tiles <= 768 ? 3 : 4;
  auto k = nt == 1 ? k_bf16_rows_mfma<1, 1, true> : nt == 2 ? k_bf16_rows_mfma<2, 1, true>
         : nt == 3 ? k_bf16_rows_mfma<3, 1, true> : k_bf16_rows_mfma<4, 1, true>;
  hipLaunchKernelGGL(k, dim3((unsigned)egroups, (unsigned)((T + 16 * nt - 1) / (16 * nt))),
                     dim3(256), 0, st, score, x, G, H, E, 0, 0, T, choice, bias);
  return dsv4g_check_launch("router_scores");
}

extern "C" {

int dsv4g_quant_fp8_act(float *qx, float *qscale, const float *x, int n, int nvec,
                        void *stream) {
  if (n <= 0 || nvec <= 0) return dsv4g_fail(DSV4G_EINVAL, "quant_fp8_act: bad size");
  dim3 grid((n + 127) / 128, nvec);
  hipLaunchKernelGGL(k_quant_fp8_act, grid, dim3(64), 0, (hipStream_t)stream, qx, qscale,
                     x, n);
  return dsv4g_check_launch("quant_fp8_act");
}

int dsv4g_dequant_fp4(float *out, const uint8_t *W, const uint8_t *S, int rows, int cols,
                      void *stream) {
  hipLaunchKernelGGL(k_dequant_fp4, dim3(1024), dim3(256), 0, (hipStream_t)stream, out, W,
                     S, rows, cols);
  return dsv4g_check_launch("dequant_fp4");
}

int dsv4g_dequant_fp8(float *out, const uint8_t *W, const uint8_t *S, int rows, int cols,
                      void *stream) {
  hipLaunchKernelGGL(k_dequant_fp8, dim3(1024), dim3(256), 0, (hipStream_t)stream, out, W,
                     S, rows, cols);
  return dsv4g_check_launch("dequant_fp8");
}

static int fp4_shape_ok(int in, const char *who) {
  if (in <= 0 || in % 32 != 0 || in > 32 * 256) {
    return dsv4g_fail(DSV4G_EINVAL, "%s: FP4 input width %d must be a positive multiple of "
                                    "32 and at most 8192", who, in);
  }
  return 0;
}

static int fp8_shape_ok(int in, const char *who) {
  if (in <= 0 || in % 16 != 0 || in > FP8_MAX_IN) {
    return dsv4g_fail(DSV4G_EINVAL, "%s: FP8 input width %d must be a positive multiple of "
                                    "16 and at most %d", who, in, FP8_MAX_IN);
  }
  return 0;
}

int dsv4g_launch_gemv_fp4(const GemvArgs *a, int nvec, int nmat, void *stream) {
  if (fp4_shape_ok(a->in, "gemv_fp4")) return DSV4G_EINVAL;
  if (a->rows <= 0 || nvec <= 0) return dsv4g_fail(DSV4G_EINVAL, "gemv_fp4: bad size");
  hipStream_t st = (hipStream_t)stream;
  // passes per tile: the most that still give about 1024 workgroups (paired
  // tiles hold at least one pass of each matrix)
  const int pair = nmat == 2;
  int np = 16;
  while (np > (pair ? 2 : 1)) {
    const int tr = fp4_geom_np(a->in, np).tr, span = pair ? tr / 2 : tr;
    if ((long)((a->rows + span - 1) / span) * nvec >= 1024) break;
    np /= 2;
  }
  if (a->np) np = a->np;
  switch (np) {
    case 1: launch_fp4_t<1>(a, nvec, pair, st); break;
    case 2: launch_fp4_t<2>(a, nvec, pair, st); break;
    case 4: launch_fp4_t<4>(a, nvec, pair, st); break;
    case 8: launch_fp4_t<8>(a, nvec, pair, st); break;
    default: launch_fp4_t<16>(a, nvec, pair, st); break;
  }
  return dsv4g_check_launch("gemv_fp4");
}

// Fits (us) of the two forms of the FP8 projection for several tokens. Matrix
// unit: up to 8 blocks a row, 1.9 per block for every 512 workgroups (two on a
// CU), 1.1 for a last 256 (1024 columns: 8192 rows 12.7 to 16 tokens, 18.6 at 33;
// 32768 rows 19.5, 35, 50 for 16, 32, 33); beyond, four waves share a row tile:
// 1.15 per block of a wave, then 1.2 for every further 256 workgroups, which are
// shared out evenly while LDS takes two on a CU (4096 columns: 1024 rows 12, 8192
// rows 19, 34, 49 for 16, 32, 33 tokens; 8192 columns x 4096 rows 23, 42, 61).
static double fp8_mfma_us(int rows, int CB, int ks, int nvec, int nmat) {
  const long wgs = (rows + 64 / ks - 1L) / (64 / ks) * ((nvec + 15) / 16) * nmat;
  if (ks == 1) {
    const long last = wgs % 512;
    const double t = 4.6 + CB * (1.9 * (wgs / 512) + (last > 256 ? 1.9 : last ? 1.1 : 0.0));
    return std::max(t, 6.0);
  }
  const int q = (CB + 3) / 4;
  const bool two = fp8_mfma_lds<4>(CB) <= 80 * 1024;
  const double more = two ? std::max(wgs / 256.0 - 1, 0.0) : (double)((wgs + 255) / 256 - 1);
  return 3.7 + 1.15 * q + 1.2 * q * more;
}

// VALU: by token and million weights, a row counted to its last lane (a row of
// 128 columns busies one of its 8 lanes, of 1152 nine of 16, of 2304 18 of 32): 128
// columns x 512 rows 5.2 and 6.0 for 16 and 33 tokens; 2048 x 4096 7.0, 9.4 for 4, 8;
// 8192 x 4096 21.7, 29, 51, 96 for 5, 8, 16, 33; four tokens at a time 1024 x 32768
// 19, 29, 57 for 8, 16, 33, 384 x 32768 9.7 for 4.
static double fp8_valu_us(int rows, int CB, int sl, bool many, int nvec, int nmat) {
  const int lanes = (CB + sl - 1) / sl * sl;
  const double c = sl == 32 ? 0.035 + 0.05 * CB / lanes
                 : many     ? (sl == 16 ? 0.01 + 0.05 * CB / lanes : 0.035 + 0.0014 * CB)
                            : (sl == 16 ? 0.062 : 0.055);
  return 5 + c * 128e-6 * lanes * nvec * nmat * rows;
}

int dsv4g_launch_gemv_fp8(const GemvArgs *a, int nvec, int nmat, void *stream) {
  if (fp8_shape_ok(a->in, "gemv_fp8")) return DSV4G_EINVAL;
  if (a->rows <= 0 || nvec <= 0) return dsv4g_fail(DSV4G_EINVAL, "gemv_fp8: bad size");
  hipStream_t st = (hipStream_t)stream;
  // lanes per row: one 128-column block per lane up to 32 blocks (more
  // workgroups, so more weight loads in flight: 4096-wide rows 6.3 -> 5.4 us
  // at 1024 and 512 rows), two beyond (8192-wide rows: one block per lane
  // measured no faster at one token and slower at five), at least 8 lanes
  // per row (shorter rows: a lane per block, the rest idle)
  // tokens four at a time only when the row tiles alone fill the GPU (a
  // smaller matrix runs one token per workgroup, all tokens in parallel)
  const int CB = (a->in + 127) / 128;
  const int sl = CB <= 8 ? 8 : CB <= 16 ? 16 : 32;
  // (and the four tokens' activations fit LDS beside the rest: in <= 2048)
  const bool many = nvec > 1 && a->in <= 2048 &&
                    (long)(a->rows + 256 / sl - 1) / (256 / sl) * nmat >= 1024;
  // several tokens on the matrix unit where it is the faster
  if (nvec > 1 && a->in % 128 == 0) {
    const int ks = CB > 8 ? 4 : 1;
    if (fp8_mfma_us(a->rows, CB, ks, nvec, nmat) < fp8_valu_us(a->rows, CB, sl, many, nvec, nmat)) {
      DSV4G_TRY(ks == 4 ? launch_fp8_proj_mfma<4>(a, nvec, nmat, st)
                        : launch_fp8_proj_mfma<1>(a, nvec, nmat, st));
      return dsv4g_check_launch("gemv_fp8");
    }
  }
  switch (sl * (many ? 10 : 1)) {
    case 8: launch_fp8_proj<8, 1>(a, nvec, nmat, st); break;
    case 16: launch_fp8_proj<16, 1>(a, nvec, nmat, st); break;
    case 80: launch_fp8_proj<8, 4>(a, nvec, nmat, st); break;
    case 160: launch_fp8_proj<16, 4>(a, nvec, nmat, st); break;
    default: launch_fp8_proj<32, 1>(a, nvec, nmat, st); break;
  }
  return dsv4g_check_launch("gemv_fp8");
}

int dsv4g_gemv_fp4_q(float *y, const float *qx, const float *qscale, const uint8_t *W,
                     const uint8_t *S, int in, int rows, void *stream) {
  GemvArgs a = {};
  a.y[0] = y;
  a.qx = qx;
  a.qscale = qscale;
  a.W[0] = W;
  a.S[0] = S;
  a.in = in;
  a.rows = rows;
  a.round_out = 1;
  return dsv4g_launch_gemv_fp4(&a, 1, 1, stream);
}

int dsv4g_gemv_fp4_pair_q(float *y0, float *y1, const float *qx, const float *qscale,
                          const uint8_t *W0, const uint8_t *S0, const uint8_t *W1,
                          const uint8_t *S1, int in, int rows, void *stream) {
  GemvArgs a = {};
  a.y[0] = y0;
  a.y[1] = y1;
  a.qx = qx;
  a.qscale = qscale;
  a.W[0] = W0;
  a.S[0] = S0;
  a.W[1] = W1;
  a.S[1] = S1;
  a.in = in;
  a.rows = rows;
  a.round_out = 1;
  return dsv4g_launch_gemv_fp4(&a, 1, 2, stream);
}

int dsv4g_gemv_fp4_batch_q(float *y, const float *qx, const float *qscale, int batch,
                           const uint8_t *W, const uint8_t *S, int in, int rows,
                           void *stream) {
  GemvArgs a = {};
  a.y[0] = y;
  a.qx = qx;
  a.qscale = qscale;
  a.W[0] = W;
  a.S[0] = S;
  a.in = in;
  a.rows = rows;
  a.round_out = 1;
  a.y_stride = rows;
  a.qx_stride = in;
  a.qs_stride = (in + 127) / 128;
  return dsv4g_launch_gemv_fp4(&a, batch, 1, stream);
}

int dsv4g_gemv_fp8_q(float *y, const float *qx, const float *qscale, const uint8_t *W,
                     const uint8_t *S, int in, int out, int round_out, void *stream) {
  GemvArgs a = {};
  a.y[0] = y;
  a.qx = qx;
  a.qscale = qscale;
  a.W[0] = W;
  a.S[0] = S;
  a.in = in;
  a.rows = out;
  a.round_out = round_out;
  return dsv4g_launch_gemv_fp8(&a, 1, 1, stream);
}

int dsv4g_gemv_fp8_pair_q(float *y0, float *y1, const float *qx, const float *qscale,
                          const uint8_t *W0, const uint8_t *S0, const uint8_t *W1,
                          const uint8_t *S1, int in, int out, void *stream) {
  GemvArgs a = {};
  a.y[0] = y0;
  a.y[1] = y1;
  a.qx = qx;
  a.qscale = qscale;
  a.W[0] = W0;
  a.S[0] = S0;
  a.W[1] = W1;
  a.S[1] = S1;
  a.in = in;
  a.rows = out;
  a.round_out = 1;
  return dsv4g_launch_gemv_fp8(&a, 1, 2, stream);
}

int dsv4g_gemv_fp8_batch_q(float *y, const float *qx, const float *qscale, int batch,
                           const uint8_t *W, const uint8_t *S, int in, int out,
                           int round_out, void *stream) {
  GemvArgs a = {};
  a.y[0] = y;
  a.qx = qx;
  a.qscale = qscale;
  a.W[0] = W;
  a.S[0] = S;
  a.in = in;
  a.rows = out;
  a.round_out = round_out;
  a.y_stride = out;
  a.qx_stride = in;
  a.qs_stride = (in + 127) / 128;
  return dsv4g_launch_gemv_fp8(&a, batch, 1, stream);
}

int dsv4g_gemv_bf16(float *y, const float *x, const uint16_t *W, int in, int out,
                    int round_out, int batch, void *stream) {
  if (in <= 0 || out <= 0 || batch <= 0) return dsv4g_fail(DSV4G_EINVAL, "gemv_bf16: bad size");
  const size_t xb = (size_t)batch * in * 4;
  if (in % 64 == 0 && ((uintptr_t)x & 15) == 0 && (size_t)64 * in * 2 < 0xFFFF0000u) {
    // runs of up to 64 tokens through the matrix unit's chains, or the tiled
    // chains where those are the faster (tiled_width); rows too wide for a run's x
    // within one buffer range go through the tiled chains two tokens at a time
    const bool wide = (size_t)64 * in * 4 >= 0xFFFF0000u;
    for (int t0 = 0; t0 < batch;) {
      const int n = std::min(batch - t0, wide ? 2 : 64);
      if (wide || in <= tiled_width(n, out)) {
        auto k = n == 1 ? k_bf16_rows_tiled<1> : n == 2 ? k_bf16_rows_tiled<2>
               : n == 3 ? k_bf16_rows_tiled<3> : n == 4 ? k_bf16_rows_tiled<4>
                        : k_bf16_rows_tiled<8>;
        hipLaunchKernelGGL(k, dim3((out + 63) / 64), dim3(64), 0, (hipStream_t)stream, y, x, W, in,
                           out, round_out, t0);
      } else {
        launch_rows_mfma(y, x, W, in, out, round_out, t0, n, (hipStream_t)stream);
      }
      DSV4G_TRY(dsv4g_check_launch("gemv_bf16"));
      t0 += n;
    }
    return 0;
  }
  if (in % 8 == 0 && xb <= RC_XBYTES && (size_t)64 * in * 2 < 0xFFFF0000u &&
      ((uintptr_t)x & 15) == 0) {
    RowChainArgs a = {};
    a.y = y;
    a.x = x;
    a.W = reinterpret_cast<const uint8_t *>(W);
    a.in = in;
    a.rows = out;
    a.batch = batch;
    a.round_out = round_out;
    a.y_stride = (size_t)out;
    a.x_stride = (size_t)in;
    const dim3 grid((out + 63) / 64);
    if (batch == 1)
      hipLaunchKernelGGL((k_rowchain<RC_BF16, 1>), grid, dim3(64), xb, (hipStream_t)stream, a);
    else if (batch <= 4)
      hipLaunchKernelGGL((k_rowchain<RC_BF16, 4>), grid, dim3(64), xb, (hipStream_t)stream, a);
    else if (batch <= 8)
      hipLaunchKernelGGL((k_rowchain<RC_BF16, 8>), grid, dim3(64), xb, (hipStream_t)stream, a);
    else
      hipLaunchKernelGGL((k_rowchain<RC_BF16, 33>), grid, dim3(64), xb, (hipStream_t)stream, a);
    return dsv4g_check_launch("gemv_bf16");
  }
  dim3 grid((out + 63) / 64, batch);
  hipLaunchKernelGGL(k_gemv_bf16, grid, dim3(64), 0, (hipStream_t)stream, y, x, W, in, out,
                     round_out, (size_t)out, (size_t)in);
  return dsv4g_check_launch("gemv_bf16");
}

int dsv4g_argmax(int *idx, const float *logits, int vocab, int n, size_t stride,
                 void *stream) {
  if (!idx || !logits || vocab <= 0 || n <= 0 || stride < (size_t)vocab)
    return dsv4g_fail(DSV4G_EINVAL, "argmax: bad arguments");
  // The threads that a row fills: clamped loads cost their issue, and idle waves
  // their start (8192 rows of 1000: 66 us with 16 waves of 8 loads, 9 with 4 of 1;
  // of 64: 66 and 4.4). Rows to 16384 take 4 waves up to four times round: 8192
  // rows of 16384 88 us against 95, one 3.4 against 4.8.
  const int kind = vocab <= 256 ? 0 : vocab <= 1024 ? 1 : vocab <= 16384 ? 2 : 3;
  auto k = kind == 0 ? k_argmax<64, 1> : kind == 1 ? k_argmax<256, 1>
         : kind == 2 ? k_argmax<256, 4> : k_argmax<1024, 8>;
  hipLaunchKernelGGL(k, dim3((unsigned)n), dim3(kind == 0 ? 64 : kind == 3 ? 1024 : 256), 0,
                     (hipStream_t)stream, idx, logits, vocab, stride);
  return dsv4g_check_launch("argmax");
}

int dsv4g_gemv_fp8_float(float *y, const float *x, const uint8_t *W, const float *wscale,
                         int in, int rows, int block, int mode, void *stream) {
  if (in <= 0 || rows <= 0 || block <= 0)
    return dsv4g_fail(DSV4G_EINVAL, "gemv_fp8_float: bad size");
  // split chains where the row is long, or too ragged for the product chains
  // (2048 rows of 3008 columns 14 us against 17, of 2048 12.6 against 12.0, of
  // 1024 11 against 7.5; of 2064 12.5 against 22), as long as they are the faster
  // beside a lane per row by these fits (us): the split's rounds of workgroups
  // against one row's time, which hardly grows with the rows (2048, 4096, 8192,
  // 32768 rows of 1040 columns, split 10.9, 15.3, 26, 82 and a lane per row 12.2,
  // 12.1, 12.1, 15; of 4096 16.9, 27, 50, 168 and 39.6, 39.7, 42, 46)
  const bool xs = mode == 0 && block % 64 == 0;  // k_rowchain's scaled x in LDS
  const double split = 6 + rows / 1024.0 * (1.5 + 0.9e-3 * in);
  const double lanes = xs ? 2.9 + 9.0e-3 * in : 2.6 + 11.4e-3 * in;
  if (in % 16 == 0 && (in > PC_MAXIN || (in % 32 && in >= PS_MININ)) && in <= PS_MAXIN &&
      block % 16 == 0 && ((uintptr_t)x & 15) == 0 && split < lanes) {
    // more than the default 64 KB of LDS (a host-side setting of the kernel)
    auto k = mode == 0 ? k_fp8_prodsplit<0> : k_fp8_prodsplit<1>;
    DSV4G_HIP(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)ps_lds(PS_MAXIN)));
    hipLaunchKernelGGL(k, dim3((unsigned)((rows + PS_ROWS - 1) / PS_ROWS)), dim3(64 * PS_ROWS),
                       ps_lds(in), (hipStream_t)stream, y, x, W, wscale, in, rows, block);
    return dsv4g_check_launch("gemv_fp8_float");
  }
  if (in % 32 == 0 && in <= PC_MAXIN && block % 16 == 0 && ((uintptr_t)x & 15) == 0) {
    const size_t lds = ((size_t)in + (size_t)PC_ROWS * (in + 4) + (in + block - 1) / block) * 4;
    const void *fn = mode == 0 ? (const void *)k_fp8_prodchain<0> : (const void *)k_fp8_prodchain<1>;
    // more than the default 64 KB of LDS (a host-side setting of the kernel)
    DSV4G_HIP(hipFuncSetAttribute(
        fn, hipFuncAttributeMaxDynamicSharedMemorySize,
        (int)(((size_t)PC_MAXIN + (size_t)PC_ROWS * (PC_MAXIN + 4) + PC_MAXIN / 16) * 4)));
    const dim3 grid((unsigned)((rows + PC_ROWS - 1) / PC_ROWS));
    if (mode == 0)
      hipLaunchKernelGGL(k_fp8_prodchain<0>, grid, dim3(256), lds, (hipStream_t)stream, y, x, W,
                         wscale, in, rows, block);
    else
      hipLaunchKernelGGL(k_fp8_prodchain<1>, grid, dim3(256), lds, (hipStream_t)stream, y, x, W,
                         wscale, in, rows, block);
    return dsv4g_check_launch("gemv_fp8_float");
  }
  if (in % 16 == 0 && block % 16 == 0 && (size_t)in * 4 * 2 <= RC_XBYTES &&
      ((uintptr_t)x & 15) == 0) {
    RowChainArgs a = {};
    a.y = y;
    a.x = x;
    a.W = W;
    a.wscale = wscale;
    a.in = in;
    a.rows = rows;
    a.block = block;
    a.batch = 1;
    const dim3 grid((rows + 63) / 64);
    const size_t xb = (size_t)in * 4 + (size_t)(64 / block + 2) * ((in + block - 1) / block) * 4;
    if (xs)
      hipLaunchKernelGGL((k_rowchain<RC_FP8_XS, 1>), grid, dim3(64), xb, (hipStream_t)stream, a);
    else if (mode == 0)
      hipLaunchKernelGGL((k_rowchain<RC_FP8_X, 1>), grid, dim3(64), xb, (hipStream_t)stream, a);
    else
      hipLaunchKernelGGL((k_rowchain<RC_FP8_T, 1>), grid, dim3(64), xb, (hipStream_t)stream, a);
    return dsv4g_check_launch("gemv_fp8_float");
  }
  hipLaunchKernelGGL(k_gemv_fp8_float, dim3((rows + 63) / 64), dim3(64), 0,
                     (hipStream_t)stream, y, x, W, wscale, in, rows, block, mode);
  return dsv4g_check_launch("gemv_fp8_float");
}

int dsv4g_gemv_fp4_float(float *y, const float *qx, const float *qscale, const uint8_t *W,
                         const float *wscale, int in, int rows, int group, void *stream) {
  if (in <= 0 || rows <= 0 || group <= 0)
    return dsv4g_fail(DSV4G_EINVAL, "gemv_fp4_float: bad size");
  hipLaunchKernelGGL(k_gemv_fp4_float, dim3((rows + 63) / 64), dim3(64), 0,
                     (hipStream_t)stream, y, qx, qscale, W, wscale, in, rows, group);
  return dsv4g_check_launch("gemv_fp4_float");
}

int dsv4g_quant_fp4_rows(uint8_t *packed, uint8_t *scales, const float *w, int rows, int cols,
                         void *stream) {
  if (rows <= 0 || cols <= 0 || cols % 32)
    return dsv4g_fail(DSV4G_EINVAL, "quant_fp4_rows: cols must be a multiple of 32");
  const size_t n = (size_t)rows * (cols / 32);
  hipLaunchKernelGGL(k_quant_fp4_rows, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, packed, scales, w, rows, cols);
  return dsv4g_check_launch("quant_fp4_rows");
}

int dsv4g_quant_fp8_blocks(uint8_t *codes, void *scales, const float *w, int rows, int cols,
                           int mode, void *stream) {
  if (rows <= 0 || cols <= 0) return dsv4g_fail(DSV4G_EINVAL, "quant_fp8_blocks: bad size");
  const int nb = ((rows + 127) / 128) * ((cols + 127) / 128);
  hipLaunchKernelGGL(k_quant_fp8_blocks, dim3(nb), dim3(256), 0, (hipStream_t)stream, codes,
                     scales, w, rows, cols, mode);
  return dsv4g_check_launch("quant_fp8_blocks");
}

}  // extern "C"
