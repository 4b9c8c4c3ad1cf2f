// Implicit-GEMM convolution for grids that cannot fill the chip (one image or a few, deep
// maps, the classifier's GEMV) on gfx950 fp16 MFMA: the K range is split over the waves of a
// work-group, and no barrier stands in the K loop.
//
// Same math and operands as conv_igemm_kernel (conv_mfma.hip): M = output pixels of all
// images, N = output channels, K = (ky, kx, ci) in 8-channel pieces, weights in the
// implicit-GEMM packing.  What bounds such a conv is latency: with 128-pixel tiles a 20x20
// map is four work-groups that each walk the whole K range step by step behind barriers, and
// a split over work-groups pays for fp32 partials in memory and a second launch.  Here a
// work-group owns 32 TM pixels x 32 TN channels and each of its NW waves a contiguous 1 / NW
// of the K range, walked in chunks of 32 channels: D chunks of both operands are in flight by
// LDS DMA into the wave's own part of D stages, so no barrier stands in the K loop, and the
// waves' partial sums meet in LDS at the end, added in wave order (results do not depend on
// scheduling).  Operands go through LDS although each is read once: a fragment loaded straight
// from the row-major operands touches 64 cache lines per instruction (one per lane), which
// bound the first version of this kernel, while a copy of 16 rows x 64 bytes touches 16.
// 256->256 3x3 at 20x20, one image: 19.1 us on the LDS-patch kernel, 12.0 us with fragments
// from memory, 7.4 us so; 128->256 3x3 stride 2 at 40x40: 19.9 -> 5.0 us; the 576->1024->1000
// classifier, both layers: 29.3 -> 10.1 us (about 5 us of each figure is the call itself).
#include "conv_common.hpp"
#include "kernels.hpp"

#include <cstdio>
#include <stdexcept>

namespace ivh {

namespace {
typedef __attribute__((address_space(3))) void lds_void;
// 64 lanes x 16 bytes from a buffer to consecutive LDS pieces at `lds` (wave uniform)
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, _Float16 * lds, unsigned voff)
{
  // the offset is computed here for every lane: left to itself the compiler splits a copy into
  // one for the lanes inside the image and one for the others
  __asm__ volatile("" : "+v"(voff));
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)lds, 16, (int)voff, 0, 0, 0);
}
}  // namespace

// K1: 1x1 (a chunk is a channel range of one pixel).  RAG: Cin % 8 != 0 (the last piece of a
// tap is masked).  UP: the upsample-concat input of conv_igemm_kernel (K1 only).
// D: chunks in flight per wave.
template <int TM, int TN, int NW, int D, bool K1, bool RAG, bool UP>
__global__ void __launch_bounds__(64 * NW) conv_small_kernel(const ConvParams p)
{
  using F = Mf<32>;
  typedef F::acc_t acc_t;
  constexpr int NT = 64 * NW, NB = TM * TN;
  constexpr int WR = (TM + TN) * 1024;      // halves of a wave's region of a stage: 32-row tiles of 32 channels
  constexpr int NI = 2 * (TM + TN);         // copies per chunk
  static_assert(D >= 2 && D <= 4, "stages");
  // one LDS object per stage: the compiler's wait analysis then sees that reading a stage does
  // not depend on the copies in flight into the others
  __shared__ __attribute__((aligned(16))) _Float16 S0[NW * WR];
  __shared__ __attribute__((aligned(16))) _Float16 S1[NW * WR];
  __shared__ __attribute__((aligned(16))) _Float16 S2[D > 2 ? NW * WR : 8];
  __shared__ __attribute__((aligned(16))) _Float16 S3[D > 3 ? NW * WR : 8];
  __shared__ __attribute__((aligned(16))) float4 red[NW * NB * 4 * 64];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int HWo = p.Ho * p.Wo;
  const unsigned M = (unsigned)p.batch * HWo;  // below 2^30 (small_views_ok)
  // channel tiles of one pixel tile, which gather the same input, stay on one XCD
  const int ny = (p.Cout + 32 * TN - 1) / (32 * TN);
  const int lin = xcd_tile(blockIdx.x, gridDim.x);
  const int bx = lin / ny, by = lin - bx * ny;
  const unsigned m0 = (unsigned)bx * (32 * TM);
  const int n0 = by * (32 * TN);

  const long x_last = (long)(p.batch - 1) * p.x.img + ((long)p.H * p.W - 1) * p.x.cs + p.cin8;
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<__half *>(p.x.ptr), (short)0, (int)(x_last * 2), kBufDword3);
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<__half *>(p.w + (long)n0 * p.kpad), (short)0, 32 * TN * p.kpad * 2, kBufDword3);
  const long u_last = UP ? (long)(p.batch - 1) * p.xu.img + ((long)(p.H >> 1) * (p.W >> 1) - 1) * p.xu.cs + p.cu : 0;
  const __amdgpu_buffer_rsrc_t ur = __builtin_amdgcn_make_buffer_rsrc(
      UP ? const_cast<__half *>(p.xu.ptr) : const_cast<__half *>(p.x.ptr), (short)0, (int)(u_last * 2), kBufDword3);

  // A copy moves 16 rows (pixels or weight rows) of 32 channels: lane i brings row i / 4's
  // piece (i % 4) ^ (row / 4 % 4) to LDS piece i, so the fragment reads below -- 32 rows at one
  // channel offset -- fall on every bank (rows of 64 bytes: without the exclusive-or four rows
  // apart share a slot).
  const int crow = lane >> 2, cpc = (lane & 3) ^ ((lane >> 4) & 3);
  int base[2 * TM], iy0[K1 ? 1 : 2 * TM], ix0[K1 ? 1 : 2 * TM], uoff[UP ? 2 * TM : 1];
  bool in[2 * TM];
#pragma unroll
  for (int t = 0; t < 2 * TM; ++t) {
    const unsigned pm = m0 + t * 16 + crow;
    in[t] = pm < M;
    const unsigned pc = in[t] ? pm : 0;
    const int b = (int)fastdiv(pc, p.dv_hwo), hw = (int)pc - b * HWo;
    const int oy = (int)fastdiv((unsigned)hw, p.dv_wo), ox = hw - oy * p.Wo;
    const int iy = oy * p.S - p.P, ix = ox * p.S - p.P;
    base[t] = b * (int)p.x.img + (iy * p.W + ix) * p.x.cs;
    if constexpr (K1) {  // P > 0: border pixels read zeros
      in[t] = in[t] && (unsigned)iy < (unsigned)p.H && (unsigned)ix < (unsigned)p.W;
      if constexpr (UP) uoff[t] = b * (int)p.xu.img + ((oy >> 1) * (p.W >> 1) + (ox >> 1)) * p.xu.cs;
    } else {
      iy0[t] = in[t] ? iy : -0x4000000;  // never inside the image
      ix0[t] = ix;
    }
  }

  // this wave's chunks of four pieces, and the (tap, channel) of the lane's piece in the next
  // chunk copied; pieces past the last tap read zeros on both sides
  const int taps = K1 ? 1 : p.K * p.K;
  const int nch = (taps * p.cin8 + 31) / 32, per = (nch + NW - 1) / NW;
  const int c0 = wave * per, c1 = c0 + per < nch ? c0 + per : nch;
  const int dq = K1 ? 0 : 32 / p.cin8, dr = 32 - dq * p.cin8;
  const unsigned kmul = K1 ? 0 : (65536u + p.K - 1) / p.K;  // tap / K as in conv_igemm_kernel
  int ci = c0 * 32 + cpc * 8, tap = 0;
  if constexpr (!K1) {
    tap = ci / p.cin8;
    ci -= tap * p.cin8;
  }
  unsigned wk = (unsigned)(c0 * 64 + cpc * 16);  // byte offset of the piece in a weight row
  const unsigned wrow = (unsigned)(crow * p.kpad * 2), wstep = (unsigned)(16 * p.kpad * 2), wend = (unsigned)(p.kpad * 2);
  auto copy = [&](_Float16 * st, int c) __attribute__((always_inline)) {
    _Float16 * const a = st + wave * WR;
    const int ky = K1 ? 0 : (int)(((unsigned)tap * kmul) >> 16), kx = K1 ? 0 : tap - ky * p.K;
    const int toff = K1 ? ci : (ky * p.W + kx) * p.x.cs + ci;
    const bool up = UP && c * 32 < p.cu;  // p.cu is a whole number of chunks
#pragma unroll
    for (int t = 0; t < 2 * TM; ++t) {
      const bool ok = K1 ? in[t] && ci < p.cin8
                         : tap < taps && (unsigned)(iy0[K1 ? 0 : t] + ky) < (unsigned)p.H && (unsigned)(ix0[K1 ? 0 : t] + kx) < (unsigned)p.W;
      if (up) dma16(ur, a + t * 512, ok ? (unsigned)((uoff[UP ? t : 0] + ci) * 2) : kBufOOB);
      else dma16(xr, a + t * 512, ok ? (unsigned)((base[t] + toff) * 2) : kBufOOB);
    }
#pragma unroll
    for (int t = 0; t < 2 * TN; ++t)
      dma16(wr, a + (2 * TM + t) * 512, wk < wend ? wrow + t * wstep + wk : kBufOOB);
    wk += 64;
    ci += dr;
    if constexpr (!K1) {
      tap += dq;
      if (ci >= p.cin8) {
        ci -= p.cin8;
        ++tap;
      }
    }
  };

  // fragment of slice j of a chunk: row lane % 32, piece 2 j + lane / 32
  const int frow = lane & 31, fsw = (frow >> 2) & 3, fh = lane >> 5;
  const int foff0 = frow * 32 + ((fh ^ fsw) * 8), foff1 = frow * 32 + (((2 + fh) ^ fsw) * 8);
  int fci0 = 0, fci1 = 0;  // RAG: channel of the fragment's piece
  const int fstep = RAG ? 32 % p.cin8 : 0;
  if constexpr (RAG) {
    fci0 = (c0 * 32 + fh * 8) % p.cin8;
    fci1 = (c0 * 32 + 16 + fh * 8) % p.cin8;
  }
  acc_t acc[TN][TM];
#pragma unroll
  for (int a = 0; a < TN; ++a)
#pragma unroll
    for (int b = 0; b < TM; ++b)
#pragma unroll
      for (int v = 0; v < F::NV; ++v) acc[a][b][v] = 0.0f;
  auto mma = [&](const _Float16 * st) __attribute__((always_inline)) {
    const _Float16 * const a = st + wave * WR;
    h8 fa[2][TN], fb[2][TM];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) fb[j][tm] = *reinterpret_cast<const h8 *>(a + tm * 1024 + (j ? foff1 : foff0));
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) fa[j][tn] = *reinterpret_cast<const h8 *>(a + (TM + tn) * 1024 + (j ? foff1 : foff0));
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if constexpr (RAG) {
        u16x8 keep;
#pragma unroll
        for (int e = 0; e < 8; ++e) keep[e] = (j ? fci1 : fci0) + e < p.Cin ? (unsigned short)0xffff : (unsigned short)0;
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) fb[j][tm] = __builtin_bit_cast(h8, __builtin_bit_cast(u16x8, fb[j][tm]) & keep);
      }
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) acc[tn][tm] = F::mma(fa[j][tn], fb[j][tm], acc[tn][tm]);
    }
    if constexpr (RAG) {
      fci0 += fstep;
      if (fci0 >= p.cin8) fci0 -= p.cin8;
      fci1 += fstep;
      if (fci1 >= p.cin8) fci1 -= p.cin8;
    }
  };
  auto stage = [&](auto I) __attribute__((always_inline)) -> _Float16 * {
    constexpr int i = decltype(I)::value;
    if constexpr (i == 0) return S0;
    else if constexpr (i == 1) return S1;
    else if constexpr (i == 2) return S2;
    else return S3;
  };
  // The wave reads only what it copied itself, so no barrier stands in the K loop: chunk c has
  // landed when at most the later chunks' copies are outstanding, and its stage is copied over
  // once its fragments are in registers.
  static_for<0, D>([&](auto I) __attribute__((always_inline)) {
    if (c0 + decltype(I)::value < c1) copy(stage(I), c0 + decltype(I)::value);
  });
  for (int c = c0; c < c1; c += D) {
    static_for<0, D>([&](auto I) __attribute__((always_inline)) {
      constexpr int i = decltype(I)::value;
      if (c + i < c1) {
        if (c + i + D <= c1) __builtin_amdgcn_s_waitcnt(vm_wait((D - 1) * NI));
        else __builtin_amdgcn_s_waitcnt(kVmWait0);  // the last D chunks were copied together
        __asm__ volatile("" ::: "memory");
        mma(stage(I));
        if (c + i + D < c1) {
          __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          copy(stage(I), c + i + D);
        }
      }
    });
  }

  // partial sums to LDS, [wave][block][4-channel run][lane]
#pragma unroll
  for (int tn = 0; tn < TN; ++tn)
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
      for (int v4 = 0; v4 < 4; ++v4)
        red[((wave * NB + tn * TM + tm) * 4 + v4) * 64 + lane] =
            make_float4(acc[tn][tm][4 * v4], acc[tn][tm][4 * v4 + 1], acc[tn][tm][4 * v4 + 2], acc[tn][tm][4 * v4 + 3]);
  __syncthreads();

  // each lane finishes runs of four channels of one pixel: sum, bias, activation, one rounding,
  // then the residual (rounded again), as the fused epilogue of the other kernels
  const _Float16 * rbase = reinterpret_cast<const _Float16 *>(p.r.ptr);
  _Float16 * ybase = reinterpret_cast<_Float16 *>(p.y.ptr);
  const bool yvec = ((p.y.cs | (int)(reinterpret_cast<uintptr_t>(ybase) >> 1) | (int)p.y.img) & 3) == 0;
  const bool rvec = ((p.r.cs | (int)(reinterpret_cast<uintptr_t>(rbase) >> 1) | (int)p.r.img) & 3) == 0;
#pragma unroll
  for (int it0 = 0; it0 < NB * 256; it0 += NT) {
    const int it = it0 + tid;
    if (NB * 256 % NT && it >= NB * 256) break;
    const int blk = it >> 8, l = it & 63, v4 = (it >> 6) & 3;
    const int tn = blk / TM, tm = blk - tn * TM;
    const unsigned pm = m0 + tm * 32 + (l & 31);
    const int co = n0 + tn * 32 + F::row(l, 4 * v4);
    if (pm >= M || co >= p.Cout) continue;
    const int b = (int)fastdiv(pm, p.dv_hwo), hw = (int)pm - b * HWo;
    const int nv = p.Cout - co < 4 ? p.Cout - co : 4;
    h4 rv = h4{};
    if (rbase) {
      const _Float16 * rp = rbase + (long)b * p.r.img + (long)hw * p.r.cs + co;
      if (rvec && nv == 4) rv = *reinterpret_cast<const h4 *>(rp);
      else
        for (int k = 0; k < nv; ++k) rv[k] = rp[k];
    }
    float4 s = red[it];
#pragma unroll
    for (int w = 1; w < NW; ++w) {
      const float4 t = red[w * NB * 256 + it];
      s.x += t.x;
      s.y += t.y;
      s.z += t.z;
      s.w += t.w;
    }
    float o[4] = {s.x, s.y, s.z, s.w};
    if (p.bias) {
      const float4 b4 = *reinterpret_cast<const float4 *>(p.bias + co);
      o[0] += b4.x;
      o[1] += b4.y;
      o[2] += b4.z;
      o[3] += b4.w;
    }
    h4 hv;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float v = o[k];
      switch (p.act) {
      case kActSiLU: v = act_fast<kActSiLU>(v); break;
      case kActReLU: v = act_fast<kActReLU>(v); break;
      case kActHSwish: v = act_fast<kActHSwish>(v); break;
      case kActHSigmoid: v = act_fast<kActHSigmoid>(v); break;
      case kActSigmoid: v = act_fast<kActSigmoid>(v); break;
      default: break;
      }
      hv[k] = round_f16(v);
    }
    if (rbase) {
#pragma unroll
      for (int k = 0; k < 4; ++k) hv[k] = (_Float16)((float)hv[k] + (float)rv[k]);
    }
    _Float16 * yp = ybase + (long)b * p.y.img + (long)hw * p.y.cs + co;
    if (yvec && nv == 4) *reinterpret_cast<h4 *>(yp) = hv;
    else
      for (int k = 0; k < nv; ++k) yp[k] = hv[k];
  }
}

// ---------------------------------------------------------------- host side

namespace {
struct SmallCfg {
  int tm, tn, nw;
};
// tile (32-pixel and 32-channel blocks) and waves per config
constexpr SmallCfg kSmallCfg[kSmallCfgs] = {{1, 1, 8}, {1, 1, 4}, {2, 1, 8}, {2, 2, 4}};
}  // namespace

long small_grid(const ConvParams & p, int cfg)
{
  const SmallCfg & c = kSmallCfg[cfg];
  const long M = (long)p.batch * p.Ho * p.Wo;
  return (M + 32 * c.tm - 1) / (32 * c.tm) * ((p.Cout + 32 * c.tn - 1) / (32 * c.tn));
}

bool small_views_ok(const ConvParams & p)
{
  return p.G == 1 && p.x.layout == kNHWC && p.x.cs % 8 == 0 && p.x.img % 8 == 0 &&
         (reinterpret_cast<uintptr_t>(p.x.ptr) & 15) == 0 && p.y.layout == kNHWC &&
         (!p.r.ptr || p.r.layout == kNHWC) && p.K * p.K + 16 < 65536 / p.K && !p.xt && !p.xg &&
         p.kpad >= p.K * p.K * p.cin8 && (long)p.batch * p.Ho * p.Wo < (1L << 30);
}

// The smallest tile whose grid runs in one round (LDS: configs 0, 2 and 3 one work-group per
// CU, config 1 two): a tile's time is mostly the latency of its first chunks, which a second
// round pays again.  Measured on MI355X as single calls, against the kernel chosen otherwise:
//   128->192 3x3 at 40x40, batch 1 / 2 / 4 (150, 150, 300 work-groups of config 2, 3, 3):
//     6.5 vs 11.8, 10.2 vs 12.2, 19.4 vs 13.7 us
//   64->128 3x3 stride 2 at 80x80, batch 1 / 2 / 4 / 8: 4.6 vs 13.2, 5.3 vs 13.2, 8.1 vs 13.4,
//     14.8 (400 work-groups) vs 13.8 us
//   256->256 3x3 at 20x20, batch 1 / 4 / 8 / 16: 7.4 vs 19.1, 9.4 vs 19.6, 16.4 vs 20.9, 31.8
//     (400) vs 30.9 us
//   384->128 1x1 at 40x40, batch 1 / 2 / 4 / 8: 4.9 vs 11.7, 5.5 vs 11.8, 7.5 vs 11.9, 13.2
//     (400) vs 13.5 us
//   64->64 1x1 at 80x80, batch 1 / 2: 5.1 vs 5.9, 6.1 (config 3, two chunks) vs 5.6 us
// Config 0 gives eight waves a K range of at least two chunks each.  Config 3 gives its four
// waves at least one each (K > 96 in 1x1 convs; any 3x3 that gets here is longer).  1x1 at that
// end, against the DMA-fed implicit GEMM: 104->128 at 40x40, batch 4: 6.0 vs 7.8 us, 192->256 at
// 40x40, batch 2: 6.5 vs 8.2; with 33 to 64 outputs that build's smaller tile is the faster one
// (128->64 at 40x40, batch 8: 5.9 vs 5.3 us, 320->64: 7.0 vs 5.8), which the rule does not use.
int small_plan(const ConvParams & p)
{
  if (!small_views_ok(p)) return 0;
  constexpr long kCUs = 256;
  const int nch = (p.K * p.K * p.cin8 + 31) / 32;
  if (nch >= 16 && small_grid(p, 0) <= kCUs) return 1;
  if (small_grid(p, 1) <= (nch >= 24 ? kCUs : 2 * kCUs)) return 2;
  if (small_grid(p, 2) <= kCUs) return 3;
  if (nch >= 4 && p.Cout > 32 && small_grid(p, 3) <= kCUs) return 4;
  return 0;
}

std::string small_launch_tag(const ConvParams & p)
{
  const SmallCfg & c = kSmallCfg[p.small - 1];
  char b[96];
  snprintf(b, sizeof b, "bm=%d bn=%d waves=%d wgs=%ld%s%s", 32 * c.tm, 32 * c.tn, c.nw, small_grid(p, p.small - 1),
           (p.Cin & 7) ? " cin-ragged" : "", p.cu ? " upsample-concat" : "");
  return b;
}

template <int TM, int TN, int NW, int D>
static void launch_small_t(const ConvParams & p, int cfg, hipStream_t s)
{
  ConvParams q = p;
  q.dv_hwo = fastdiv_make((unsigned)(p.Ho * p.Wo));
  q.dv_wo = fastdiv_make((unsigned)p.Wo);
  const dim3 grid((unsigned)small_grid(p, cfg)), block(64 * NW);
  const bool rag = (p.Cin & 7) != 0;
  if (p.cu) hipLaunchKernelGGL((conv_small_kernel<TM, TN, NW, D, true, false, true>), grid, block, 0, s, q);
  else if (p.K == 1 && rag) hipLaunchKernelGGL((conv_small_kernel<TM, TN, NW, D, true, true, false>), grid, block, 0, s, q);
  else if (p.K == 1) hipLaunchKernelGGL((conv_small_kernel<TM, TN, NW, D, true, false, false>), grid, block, 0, s, q);
  else if (rag) hipLaunchKernelGGL((conv_small_kernel<TM, TN, NW, D, false, true, false>), grid, block, 0, s, q);
  else hipLaunchKernelGGL((conv_small_kernel<TM, TN, NW, D, false, false, false>), grid, block, 0, s, q);
}

void launch_conv_small(const ConvParams & p, hipStream_t s)
{
  if (!small_views_ok(p) || (p.cu && !upcat_ok(p))) throw std::runtime_error("small-grid conv geometry");
  switch (p.small - 1) {
  case 0: launch_small_t<1, 1, 8, 3>(p, 0, s); break;
  case 1: launch_small_t<1, 1, 4, 4>(p, 1, s); break;
  case 2: launch_small_t<2, 1, 8, 2>(p, 2, s); break;
  default: launch_small_t<2, 2, 4, 3>(p, 3, s); break;
  }
}

}  // namespace ivh
