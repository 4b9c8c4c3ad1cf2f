// The implicit GEMM of conv_mfma.hip fed through LDS by DMA, gfx950 fp16 MFMA: the channels-last
// 1x1 and strided convs whose grids fill the chip.
//
// Same tiles (128 pixels x 64 or 128 channels, 4 waves), operands, K order and rounding as
// conv_igemm_kernel, and so the same results with the whole K range (KG = 1).  That kernel
// carries both operands through registers into LDS: as many LDS writes as reads, 16 to 32
// registers a step.  Here buffer loads with the LDS flag copy a step of 32 channels (128 rows of 64 bytes per operand,
// swizzled as in conv_small.hip) into one of three stages, two steps ahead; a wave waits for
// its own copies of the step (a compile-time vmcnt count), one barrier publishes every wave's
// and retires the stage the next copies overwrite; the fragments are read before the next
// copies' addresses are computed, so neither waits for the other.  Outputs go from the
// accumulators to memory as 16-byte pieces of eight channels (v_permlane32_swap between the
// lane halves).
// A step of one such work-group is a serial chain of about 1000 cycles (barrier, LDS latency,
// addresses, 256 cycles of MFMA) whatever the depth of the ring (three to eight stages measured
// the same), so with at most one work-group per CU eight waves halve the K range between
// two groups with stages of their own (KG = 2) and add their sums through LDS at the end.
// Measured on MI355X as single calls, against conv_igemm_kernel: 128->256 3x3 stride 2 at 40x40,
// batch 16 / 64 (KG 2, 1): 21.2 -> 15.7, 30.5 -> 29.8 us; 64->64 at 80x80 stride 2, batch 11
// (KG 2): 11.6 -> 7.9 us; 512->256 1x1 at 20x20, batch 64 (KG 1): 18.3 -> 17.5 us; 384->128 1x1 at
// 40x40, batch 32 (KG 1): 18.7 -> 16.4 us.
#include "conv_common.hpp"
#include "kernels.hpp"

#include <stdexcept>

namespace ivh {

namespace {
typedef __attribute__((address_space(3))) void lds_void;
typedef unsigned u2 __attribute__((ext_vector_type(2)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, _Float16 * lds, unsigned voff)
{
  // the offset is computed here for every lane: left to itself the compiler splits a copy into
  // one for the lanes inside the image and one for the others
  __asm__ volatile("" : "+v"(voff));
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)lds, 16, (int)voff, 0, 0, 0);
}
constexpr int kRingD = 3;  // stages
}  // namespace

template <int ACT, int TM, int TN>
__device__ __forceinline__ void ring_epilogue(const ConvParams & p, Mf<32>::acc_t (&acc)[TN][TM], unsigned m0, int n0)
{
  using F = Mf<32>;
  const int lane = threadIdx.x & 63, HWo = p.Ho * p.Wo;
  const unsigned M = (unsigned)p.batch * HWo;
  const _Float16 * rbase = reinterpret_cast<const _Float16 *>(p.r.ptr);
  _Float16 * ybase = reinterpret_cast<_Float16 *>(p.y.ptr);
#pragma unroll
  for (int tm = 0; tm < TM; ++tm) {
    const unsigned pm = m0 + tm * 32 + (lane & 31);
    const unsigned pc = pm < M ? pm : 0;
    const int b = (int)fastdiv(pc, p.dv_hwo), hw = (int)pc - b * HWo;
    _Float16 * yp = ybase + (long)b * p.y.img + (long)hw * p.y.cs;
    const _Float16 * rp = rbase ? rbase + (long)b * p.r.img + (long)hw * p.r.cs : nullptr;
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
      for (int v8 = 0; v8 < 16; v8 += 8) {
        u2 h[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const int v4 = v8 + 4 * s;
          float4 b4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
          if (p.bias) b4 = *reinterpret_cast<const float4 *>(p.bias + n0 + tn * 32 + F::row(lane, v4));
          const float bb[4] = {b4.x, b4.y, b4.z, b4.w};
          h4 hv;
#pragma unroll
          for (int k = 0; k < 4; ++k) hv[k] = round_f16(act_fast<ACT>(acc[tn][tm][v4 + k] + bb[k]));
          h[s] = __builtin_bit_cast(u2, hv);
        }
        const auto s0 = __builtin_amdgcn_permlane32_swap(h[0][0], h[1][0], false, false);
        const auto s1 = __builtin_amdgcn_permlane32_swap(h[0][1], h[1][1], false, false);
        h8 v = __builtin_bit_cast(h8, u4{s0[0], s1[0], s0[1], s1[1]});
        const int co = n0 + tn * 32 + 2 * v8 + 8 * (lane >> 5);
        if (pm >= M || co >= p.Cout) continue;
        if (rp) {
          const h8 rv = *reinterpret_cast<const h8 *>(rp + co);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = (_Float16)((float)v[e] + (float)rv[e]);
        }
        *reinterpret_cast<h8 *>(yp + co) = v;
      }
  }
}

// K1: 1x1; UP: its upsample-concat input (conv_igemm_kernel).  KG = 2: eight waves, two groups
// of four over the halves of the K range with stages of their own.
template <int TN, int KG, bool K1, bool UP>
__global__ void __launch_bounds__(256 * KG, 2) conv_ring_kernel(const ConvParams p)
{
  using F = Mf<32>;
  typedef F::acc_t acc_t;
  constexpr int TM = 2, BN = 64 * TN, D = kRingD;
  constexpr int NI = 2 + TN;              // copies per wave and step: 32 pixel rows, 16 TN weight rows
  constexpr int SB = (128 + BN) * 32;     // halves per stage and group
  __shared__ __attribute__((aligned(16))) _Float16 S0[KG * SB];
  __shared__ __attribute__((aligned(16))) _Float16 S1[KG * SB];
  __shared__ __attribute__((aligned(16))) _Float16 S2[KG * SB];
  __shared__ __attribute__((aligned(16))) float4 red[KG > 1 ? 8 * TN * 4 * 64 : 1];  // half a wave's partial sums each

  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave = wv & 3, kg = KG > 1 ? wv >> 2 : 0;
  const int wm = wave & 1, wn = wave >> 1;
  const int HWo = p.Ho * p.Wo;
  const unsigned M = (unsigned)p.batch * HWo;
  const int ny = (p.Cout + BN - 1) / BN;
  const int lin = xcd_tile(blockIdx.x, gridDim.x);
  const int bx = lin / ny, by = lin - bx * ny;
  const unsigned m0 = (unsigned)bx * 128;
  const int n0 = by * BN;

  const long x_last = (long)(p.batch - 1) * p.x.img + ((long)p.H * p.W - 1) * p.x.cs + p.cin8;
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<__half *>(p.x.ptr), (short)0, (int)(x_last * 2), kBufDword3);
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<__half *>(p.w + (long)n0 * p.kpad), (short)0, BN * p.kpad * 2, kBufDword3);
  const long u_last = UP ? (long)(p.batch - 1) * p.xu.img + ((long)(p.H >> 1) * (p.W >> 1) - 1) * p.xu.cs + p.cu : 0;
  const __amdgpu_buffer_rsrc_t ur = __builtin_amdgcn_make_buffer_rsrc(
      UP ? const_cast<__half *>(p.xu.ptr) : const_cast<__half *>(p.x.ptr), (short)0, (int)(u_last * 2), kBufDword3);

  // copies: 16 rows of four 8-channel pieces; lane i brings row i / 4's piece
  // (i % 4) ^ (row / 4 % 4) to LDS piece i (see conv_small.hip)
  const int crow = lane >> 2, cpc = (lane & 3) ^ ((lane >> 4) & 3);
  int base[2], iy0[2], ix0[2], uoff[2];
  bool in[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const unsigned pm = m0 + wave * 32 + t * 16 + crow;
    in[t] = pm < M;
    const unsigned pc = in[t] ? pm : 0;
    const int b = (int)fastdiv(pc, p.dv_hwo), hw = (int)pc - b * HWo;
    const int oy = (int)fastdiv((unsigned)hw, p.dv_wo), ox = hw - oy * p.Wo;
    const int iy = oy * p.S - p.P, ix = ox * p.S - p.P;
    base[t] = b * (int)p.x.img + (iy * p.W + ix) * p.x.cs;
    if (K1) in[t] = in[t] && (unsigned)iy < (unsigned)p.H && (unsigned)ix < (unsigned)p.W;
    iy0[t] = in[t] ? iy : -0x4000000;  // never inside the image
    ix0[t] = ix;
    uoff[t] = UP ? b * (int)p.xu.img + ((oy >> 1) * (p.W >> 1) + (ox >> 1)) * p.xu.cs : 0;
  }
  const int taps = K1 ? 1 : p.K * p.K;
  // this group's K steps c0 .. c0 + nk - 1 (those past the range read zeros)
  const int nk = ((taps * p.cin8 + 31) / 32 + KG - 1) / KG, c0 = kg * nk;
  const int dq = K1 ? 0 : 32 / p.cin8, dr = 32 - dq * p.cin8;
  const unsigned kmul = K1 ? 0 : (65536u + p.K - 1) / p.K;
  int ci = c0 * 32 + cpc * 8, tap = 0;
  if (!K1) {
    tap = ci / p.cin8;
    ci -= tap * p.cin8;
  }
  unsigned wk = (unsigned)(c0 * 64 + cpc * 16);
  const unsigned wrow = (unsigned)((wave * 16 * TN + crow) * p.kpad * 2), wstep = (unsigned)(16 * p.kpad * 2), wend = (unsigned)(p.kpad * 2);
  auto copy = [&](_Float16 * st, int c) __attribute__((always_inline)) {
    _Float16 * const a = st + kg * SB + wave * 1024;
    const int ky = K1 ? 0 : (int)(((unsigned)tap * kmul) >> 16), kx = K1 ? 0 : tap - ky * p.K;
    const int toff = K1 ? ci : (ky * p.W + kx) * p.x.cs + ci;
    const bool up = UP && (c0 + c) * 32 < p.cu;  // p.cu is a whole number of steps
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const bool ok = K1 ? in[t] && ci < p.cin8
                         : tap < taps && (unsigned)(iy0[t] + ky) < (unsigned)p.H && (unsigned)(ix0[t] + kx) < (unsigned)p.W;
      const unsigned off = ok ? (unsigned)((up ? uoff[t] + ci : base[t] + toff) * 2) : kBufOOB;
      if (up) dma16(ur, a + t * 512, off);
      else dma16(xr, a + t * 512, off);
    }
    _Float16 * const w = st + kg * SB + 4096 + wave * (512 * TN);
#pragma unroll
    for (int t = 0; t < TN; ++t) dma16(wr, w + t * 512, wk < wend ? wrow + t * wstep + wk : kBufOOB);
    wk += 64;
    ci += dr;
    if (!K1) {
      tap += dq;
      if (ci >= p.cin8) {
        ci -= p.cin8;
        ++tap;
      }
    }
  };

  const int frow = lane & 31, fsw = (frow >> 2) & 3, fh = lane >> 5;
  const int foff[2] = {frow * 32 + ((fh ^ fsw) * 8), frow * 32 + (((2 + fh) ^ fsw) * 8)};
  acc_t acc[TN][TM];
#pragma unroll
  for (int a = 0; a < TN; ++a)
#pragma unroll
    for (int b = 0; b < TM; ++b)
#pragma unroll
      for (int v = 0; v < F::NV; ++v) acc[a][b][v] = 0.0f;
  h8 fa[2][TN], fb[2][TM];
  auto frags = [&](const _Float16 * stage0) __attribute__((always_inline)) {
    const _Float16 * const st = stage0 + kg * SB;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int tm = 0; tm < TM; ++tm) fb[j][tm] = *reinterpret_cast<const h8 *>(st + (wm * TM + tm) * 1024 + foff[j]);
#pragma unroll
      for (int tn = 0; tn < TN; ++tn) fa[j][tn] = *reinterpret_cast<const h8 *>(st + 4096 + (wn * TN + tn) * 1024 + foff[j]);
    }
  };
  auto mma = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int tn = 0; tn < TN; ++tn)
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) acc[tn][tm] = F::mma(fa[j][tn], fb[j][tm], acc[tn][tm]);
  };
  auto stage = [&](auto I) __attribute__((always_inline)) -> _Float16 * {
    constexpr int i = decltype(I)::value;
    if constexpr (i == 0) return S0;
    else if constexpr (i == 1) return S1;
    else return S2;
  };
  static_for<0, D - 1>([&](auto I) __attribute__((always_inline)) {
    if (decltype(I)::value < nk) copy(stage(I), decltype(I)::value);
  });
  for (int s = 0; s < nk; s += D) {
    static_for<0, D>([&](auto I) __attribute__((always_inline)) {
      constexpr int i = decltype(I)::value;
      if (s + i < nk) {
        // this wave's copies of step s + i have landed (up to D - 2 later steps in flight)
        if (s + i + D - 2 < nk) __builtin_amdgcn_s_waitcnt(vm_wait((D - 2) * NI));
        else __builtin_amdgcn_s_waitcnt(kVmWait0);
        __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();  // every wave's have; every wave has read step s + i - 1
        __asm__ volatile("" ::: "memory");
        // the step's fragments are on their way from LDS while the copies' addresses are computed;
        // the copies are issued between the MFMAs
        frags(stage(I));
        if (s + i + D - 1 < nk) copy(stage(std::integral_constant<int, (i + D - 1) % D>{}), s + i + D - 1);
        mma();
      }
    });
  }

  const unsigned em = m0 + wm * 64;
  const int en = n0 + wn * TN * 32;
  auto finish = [&](auto NT, acc_t (&ac)[TN][decltype(NT)::value], unsigned mf) __attribute__((always_inline)) {
    constexpr int nt = decltype(NT)::value;
    switch (p.act) {
    case kActSiLU: ring_epilogue<kActSiLU, nt, TN>(p, ac, mf, en); break;
    case kActReLU: ring_epilogue<kActReLU, nt, TN>(p, ac, mf, en); break;
    case kActHSwish: ring_epilogue<kActHSwish, nt, TN>(p, ac, mf, en); break;
    case kActHSigmoid: ring_epilogue<kActHSigmoid, nt, TN>(p, ac, mf, en); break;
    case kActSigmoid: ring_epilogue<kActSigmoid, nt, TN>(p, ac, mf, en); break;
    default: ring_epilogue<kActNone, nt, TN>(p, ac, mf, en); break;
    }
  };
  if constexpr (KG == 1) {
    finish(std::integral_constant<int, TM>{}, acc, em);
  } else {
    // group g keeps pixel block g of every wave tile and hands the other one over
    acc_t own[TN][1];
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) {
      own[tn][0] = kg ? acc[tn][1] : acc[tn][0];
      const acc_t give = kg ? acc[tn][0] : acc[tn][1];
#pragma unroll
      for (int v4 = 0; v4 < 4; ++v4)
        red[((wv * TN + tn) * 4 + v4) * 64 + lane] = make_float4(give[4 * v4], give[4 * v4 + 1], give[4 * v4 + 2], give[4 * v4 + 3]);
    }
    __syncthreads();
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
      for (int v4 = 0; v4 < 4; ++v4) {
        const float4 t = red[(((wv ^ 4) * TN + tn) * 4 + v4) * 64 + lane];
        own[tn][0][4 * v4] += t.x;
        own[tn][0][4 * v4 + 1] += t.y;
        own[tn][0][4 * v4 + 2] += t.z;
        own[tn][0][4 * v4 + 3] += t.w;
      }
    finish(std::integral_constant<int, 1>{}, own, em + kg * 32);
  }
}

// ---------------------------------------------------------------- host side

bool ring_ok(const ConvParams & p)
{
  auto vec = [](const View & v) {
    return v.layout == kNHWC && v.cs % 8 == 0 && v.img % 8 == 0 && (reinterpret_cast<uintptr_t>(v.ptr) & 15) == 0;
  };
  return p.G == 1 && p.Cin % 8 == 0 && p.cin8 == p.Cin && p.Cout % 8 == 0 && p.Cout > 32 && !p.xt &&
         !p.xg && vec(p.x) && vec(p.y) && (!p.r.ptr || vec(p.r)) && p.K * p.K + 16 < 65536 / p.K &&
         p.kpad >= p.K * p.K * p.cin8 && (long)p.batch * p.Ho * p.Wo < (1L << 30);
}

// Which implicit-GEMM convs take this kernel: its 1 or 2, else 0.  K halves (not when an image's
// sums must have one order at every batch) while every CU has at most one work-group and each
// half has at least four steps.  The whole-K build up to the resident work-groups of one
// round (three per CU at 128 channels: 384->128 1x1 at 40x40, batch 64, is 800 tiles and 35.1 us
// against 34.6 us on the 128-VGPR build of conv_igemm_kernel, four per CU); with 64 channels
// two rounds still gain (192->64 1x1 at 80x80, batch 32, 1600 tiles: 29.8 -> 27.8 us; batch 64,
// 3200 tiles: 52.7 against 53.5 us).
int ring_plan(const ConvParams & p, bool one_order)
{
  if (!ring_ok(p)) return 0;
  const int bn = igemm_bn(p.Cout);
  const long tiles = ((long)p.batch * p.Ho * p.Wo + 127) / 128 * ((p.Cout + bn - 1) / bn);
  const int nk = (p.K * p.K * p.cin8 + 31) / 32;
  if (!one_order && tiles <= 256 && nk >= 8) return 2;
  return tiles <= (bn == 128 ? 768 : 2048) ? 1 : 0;
}

template <int TN, int KG>
static void launch_ring_t(const ConvParams & q, hipStream_t s)
{
  const long M = (long)q.batch * q.Ho * q.Wo;
  const dim3 grid((unsigned)((M + 127) / 128 * ((q.Cout + 64 * TN - 1) / (64 * TN)))), block(256 * KG);
  if (q.cu) hipLaunchKernelGGL((conv_ring_kernel<TN, KG, true, true>), grid, block, 0, s, q);
  else if (q.K == 1) hipLaunchKernelGGL((conv_ring_kernel<TN, KG, true, false>), grid, block, 0, s, q);
  else hipLaunchKernelGGL((conv_ring_kernel<TN, KG, false, false>), grid, block, 0, s, q);
}

void launch_conv_ring(const ConvParams & p, hipStream_t s)
{
  if (!ring_ok(p) || (p.cu && !upcat_ok(p))) throw std::runtime_error("implicit-GEMM conv geometry");
  ConvParams q = p;
  q.dv_hwo = fastdiv_make((unsigned)(p.Ho * p.Wo));
  q.dv_wo = fastdiv_make((unsigned)p.Wo);
  if (igemm_bn(p.Cout) == 128) {
    if (p.ring == 2) launch_ring_t<2, 2>(q, s);
    else launch_ring_t<2, 1>(q, s);
  } else {
    if (p.ring == 2) launch_ring_t<1, 2>(q, s);
    else launch_ring_t<1, 1>(q, s);
  }
}

}  // namespace ivh
