// 1x1 stride-1 convs with 64 < Cout <= 128 and 128 < Cin <= 384 on large channels-last maps,
// gfx950 fp16 MFMA: weights in registers, pixels streamed through LDS by DMA, persistent.
//
// Same operands, K order, rounding and results as conv_igemm_kernel.  Bound: HBM.  As 128 x 128 tiles such a
// layer is one round of work-groups that all load, then compute, then store (800 tiles of
// 40x40 maps at batch 64), so the memory idles between the phases and each tile fetches the
// weights again.  Here two work-groups of four waves per CU walk contiguous shares of the
// 32-pixel blocks.  Each wave keeps the weights of its 32 output channels in registers
// (NSL MFMA A fragments); the blocks pass through a ring of R LDS stages, copied R - 1 blocks
// ahead as whole 128-byte rows of 64 channels (the 16-byte pieces of a row exclusive-ored with
// bits 1..3 of the pixel, so that a fragment read falls on every bank), one barrier per
// block; a block's outputs are stored while later blocks are in flight and never waited for.
// 384->128 at 40x40, batch 64: 34.0 -> 28.1 us (3.7 TB/s); 256->128 21.7 -> 18.5, 192->128 19.7 ->
// 16.6; 192->128 at 80x80, batch 32: 45.9 -> 32.7 us.
#include "conv_common.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <stdexcept>

namespace ivh {

namespace {
typedef __attribute__((address_space(3))) void lds_void;
typedef unsigned u2 __attribute__((ext_vector_type(2)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));
constexpr int kStreamR = 3;        // LDS stages
constexpr int kStreamGrid = 512;   // two work-groups per CU
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, _Float16 * lds, unsigned voff)
{
  __asm__ volatile("" : "+v"(voff));  // one copy for all lanes (see conv_small.hip)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)lds, 16, (int)voff, 0, 0, 0);
}
}  // namespace

// NCH: 64-channel chunks (Cin <= 64 NCH; channels past Cin read zeros on both sides)
template <int NCH, int ACT>
__global__ void __launch_bounds__(256) conv1x1_stream_kernel(const ConvParams p)
{
  using F = Mf<32>;
  typedef F::acc_t acc_t;
  constexpr int NSL = 4 * NCH, R = kStreamR, SB = NCH * 2048;  // halves per stage
  __shared__ __attribute__((aligned(16))) _Float16 S0[SB];
  __shared__ __attribute__((aligned(16))) _Float16 S1[SB];
  __shared__ __attribute__((aligned(16))) _Float16 S2[SB];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int HW = p.H * p.W;
  const unsigned M = (unsigned)p.batch * HW;
  const int nb = (int)((M + 31) / 32), G = gridDim.x;
  const int g = xcd_tile(blockIdx.x, G);
  const int b_lo = (int)((long)g * nb / G), n = (int)((long)(g + 1) * nb / G) - b_lo;
  if (n <= 0) return;
  const int n0 = wave * 32;

  const long x_last = (long)(p.batch - 1) * p.x.img + ((long)HW - 1) * p.x.cs + p.cin8;
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<__half *>(p.x.ptr), (short)0, (int)(x_last * 2), kBufDword3);
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<__half *>(p.w + (long)n0 * p.kpad), (short)0, 32 * p.kpad * 2, kBufDword3);
  const long y_last = (long)(p.batch - 1) * p.y.img + ((long)HW - 1) * p.y.cs + p.Cout;
  const __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc(p.y.ptr, (short)0, (int)(y_last * 2), kBufDword3);

  // a copy moves 8 pixels x 64 channels; this wave copies pixels 8 wave .. 8 wave + 7 of a
  // block: lane i brings pixel i / 8's piece (i % 8) ^ (pixel / 2 % 8) to LDS piece i
  const int cpx = wave * 8 + (lane >> 3), cpc = (lane & 7) ^ ((cpx >> 1) & 7);
  auto copy = [&](_Float16 * st, int blk) __attribute__((always_inline)) {
    const unsigned pm = (unsigned)(b_lo + blk) * 32u + cpx;
    const unsigned pc = pm < M ? pm : 0;
    const int b = (int)fastdiv(pc, p.dv_hwo), hw = (int)pc - b * HW;
    const unsigned base = (unsigned)(b * (int)p.x.img + hw * p.x.cs + cpc * 8) * 2u;
#pragma unroll
    for (int c = 0; c < NCH; ++c)
      dma16(xr, st + c * 2048 + wave * 512, pm < M && c * 64 + cpc * 8 < p.cin8 ? base + c * 128 : kBufOOB);
  };
  static_assert(R == 3, "stages");
  copy(S0, 0);
  if (n > 1) copy(S1, 1);

  h8 wf[NSL];
#pragma unroll
  for (int s = 0; s < NSL; ++s) {
    const int k = s * 16 + F::kq(lane);
    wf[s] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(
        wr, k < p.cin8 ? (unsigned)(((lane & 31) * p.kpad + k) * 2) : kBufOOB, 0, 0));
  }
  float bias[16];
#pragma unroll
  for (int v4 = 0; v4 < 16; v4 += 4) {
    float4 b4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (p.bias) b4 = *reinterpret_cast<const float4 *>(p.bias + n0 + F::row(lane, v4));
    bias[v4] = b4.x;
    bias[v4 + 1] = b4.y;
    bias[v4 + 2] = b4.z;
    bias[v4 + 3] = b4.w;
  }
  // every fragment is in its register before the loop counts outstanding copies
#pragma unroll
  for (int s = 0; s < NSL; ++s) __asm__ volatile("" : "+v"(wf[s]));
  __builtin_amdgcn_s_waitcnt(kVmWait0);

  const int frow = lane & 31, fsw = (frow >> 1) & 7, fh = lane >> 5;
  const int fbase = frow * 64;
  int foff[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) foff[j] = fbase + (((2 * j + fh) ^ fsw) * 8);
  // copies of block i are followed by those of block i + 1 and, from the second block on, by the
  // two stores of each of the last R - 1 blocks.  The counts hold only if every block issues its
  // copies before its stores: a store moved ahead of them would let that many copies still be in
  // flight when their stage is read.  The empty asm after the copies pins that order.
  constexpr int W0 = NCH, W1 = NCH + 2 * (R - 1);
  auto block = [&](int i, const _Float16 * st, _Float16 * nx) __attribute__((always_inline)) {
    if (i + 1 >= n) __builtin_amdgcn_s_waitcnt(kVmWait0);
    else if (i >= R - 1) __builtin_amdgcn_s_waitcnt(vm_wait(W1));
    else __builtin_amdgcn_s_waitcnt(vm_wait(W0));
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();  // every wave's copies; every wave has read the stage copied next
    __asm__ volatile("" ::: "memory");
    if (i + R - 1 < n) copy(nx, i + R - 1);
    __asm__ volatile("" ::: "memory");
    acc_t acc;
#pragma unroll
    for (int v = 0; v < F::NV; ++v) acc[v] = 0.0f;
#pragma unroll
    for (int s = 0; s < NSL; ++s)
      acc = F::mma(wf[s], *reinterpret_cast<const h8 *>(st + (s / 4) * 2048 + foff[s % 4]), acc);
    const unsigned pm = (unsigned)(b_lo + i) * 32u + frow;
    const unsigned pc = pm < M ? pm : 0;
    const int b = (int)fastdiv(pc, p.dv_hwo), hw = (int)pc - b * HW;
    const unsigned yo = (unsigned)(b * (int)p.y.img + hw * p.y.cs) * 2u;
#pragma unroll
    for (int v8 = 0; v8 < 16; v8 += 8) {
      u2 h[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        h4 hv;
#pragma unroll
        for (int k = 0; k < 4; ++k) hv[k] = round_f16(act_fast<ACT>(acc[v8 + 4 * t + k] + bias[v8 + 4 * t + k]));
        h[t] = __builtin_bit_cast(u2, hv);
      }
      const auto s0 = __builtin_amdgcn_permlane32_swap(h[0][0], h[1][0], false, false);
      const auto s1 = __builtin_amdgcn_permlane32_swap(h[0][1], h[1][1], false, false);
      const int co = n0 + 2 * v8 + 8 * fh;
      unsigned off = pm < M && co < p.Cout ? yo + (unsigned)co * 2u : kBufOOB;
      __asm__ volatile("" : "+v"(off));  // always one store, the counts above rely on it
      __builtin_amdgcn_raw_buffer_store_b128(u4{s0[0], s1[0], s0[1], s1[1]}, yr, off, 0, 0);
    }
  };
  for (int i = 0; i < n; i += 3) {
    block(i, S0, S2);
    if (i + 1 < n) block(i + 1, S1, S0);
    if (i + 2 < n) block(i + 2, S2, S1);
  }
}

// ---------------------------------------------------------------- host side

bool stream_ok(const ConvParams & p)
{
  auto vec = [&](const View & v, long last) {
    return v.layout == kNHWC && v.cs % 8 == 0 && v.img % 8 == 0 && (reinterpret_cast<uintptr_t>(v.ptr) & 15) == 0 &&
           ((long)(p.batch - 1) * v.img + ((long)p.H * p.W - 1) * v.cs + last) * 2 < (1L << 31);
  };
  const bool act_ok = p.act == kActNone || p.act == kActSiLU || p.act == kActReLU || p.act == kActHSwish;
  return p.K == 1 && p.S == 1 && p.P == 0 && p.G == 1 && !p.r.ptr && !p.cu && !p.xt && !p.xg && act_ok &&
         p.Cin % 8 == 0 && p.cin8 == p.Cin && p.Cin > 128 && p.Cin <= 384 && p.kpad >= p.cin8 && p.Cout % 8 == 0 &&
         p.Cout > 64 && p.Cout <= 128 && vec(p.x, p.cin8) && vec(p.y, p.Cout) &&
         (long)p.batch * p.H * p.W < (1L << 30);
}

// From four blocks per work-group on (five above 256 input channels, whose weights take longer
// to load): batch 32 / 48 / 64 at 40x40 is 1600 / 2400 / 3200 blocks, and against the
// DMA-fed implicit GEMM 256->128 takes 14.2 vs 13.0, 15.9 vs 17.2, 18.5 vs 21.6 us, 384->128
// 18.4 vs 15.6, 20.8 vs 20.7, 28.1 vs 33.8 us.  Above 384 channels one work-group fits a CU and
// nothing is gained (512->128: 40.0 vs 41.6 us; 448->104 at 33x33: 26.6 vs 21.6 us).
bool stream_plan(const ConvParams & p)
{
  const long nb = ((long)p.batch * p.H * p.W + 31) / 32;
  return stream_ok(p) && nb >= (p.Cin <= 256 ? 4 : 5) * kStreamGrid;
}

template <int NCH>
static void launch_stream_t(const ConvParams & q, hipStream_t s)
{
  const long nb = ((long)q.batch * q.H * q.W + 31) / 32;
  const dim3 grid((unsigned)std::min<long>(nb, kStreamGrid)), block(256);
  switch (q.act) {
  case kActSiLU: hipLaunchKernelGGL((conv1x1_stream_kernel<NCH, kActSiLU>), grid, block, 0, s, q); break;
  case kActReLU: hipLaunchKernelGGL((conv1x1_stream_kernel<NCH, kActReLU>), grid, block, 0, s, q); break;
  case kActHSwish: hipLaunchKernelGGL((conv1x1_stream_kernel<NCH, kActHSwish>), grid, block, 0, s, q); break;
  default: hipLaunchKernelGGL((conv1x1_stream_kernel<NCH, kActNone>), grid, block, 0, s, q); break;
  }
}

void launch_conv_stream(const ConvParams & p, hipStream_t s)
{
  if (!stream_ok(p)) throw std::runtime_error("streaming 1x1 conv geometry");
  ConvParams q = p;
  q.dv_hwo = fastdiv_make((unsigned)(p.H * p.W));
  switch ((p.cin8 + 63) / 64) {
  case 3: launch_stream_t<3>(q, s); break;
  case 4: launch_stream_t<4>(q, s); break;
  case 5: launch_stream_t<5>(q, s); break;
  default: launch_stream_t<6>(q, s); break;
  }
}

}  // namespace ivh
