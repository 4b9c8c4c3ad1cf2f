// Batched matrix product on gfx950 fp16 MFMA (v_mfma_f32_32x32x16_f16), fp32 accumulate:
// the reference's bmm (kernels/ops.cl:276-294, dispatch src/PlanModel.cpp:3935-3990), used by
// the YOLO11n C2PSA attention (q^T k over 400 tokens, v attn^T).
//
//   Y[bb][m][n] = sum_k A[bb][m][k] * B[bb][k][n]     per image, one rounding to fp16
//
// Either operand may be stored transposed -- A as [K][M] (TA), B as [N][K] (TB) -- which is
// how a permute of the last two dimensions feeding the product is folded away.
//
// Bound: HBM (the scores and probabilities of an attention are M x N and M x K with one short
// side).  Tiles of 64 x 128 or, for N <= 64, 128 x 64 outputs, every wave 32 x 64; K steps of
// 64 in LDS as [row][k] (k contiguous: the MFMA fragment layout) with the next step's pieces in
// registers meanwhile.  An operand whose k is contiguous is copied in 16-byte pieces; the
// other is read as blocks of four k by eight (four) columns, transposed in registers and written
// as 8-byte runs of k.  Rows need no alignment: pieces are loaded and stored at 2-byte
// alignment (400 tokens or 399 run alike).  The MFMA computes the tile's transpose, so a lane
// holds four neighbouring columns of a row, and the tile is staged in LDS and written as
// 16-byte row pieces.  The tiles of one matrix run on one XCD (xcd_tile), whose L2 then reads
// its operands once.  64 images of 4 heads x 400 tokens x 64: q^T k 72 -> 36 us, P v 103 -> 24 us
// (before: K steps of 32 without prefetch, 2-byte transposing LDS stores, every matrix's tiles
// over all XCDs).
#include "conv_common.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <stdexcept>

namespace ivh {

namespace {
constexpr int kBK = 64, kLDK = kBK + 8;
typedef _Float16 h8u __attribute__((ext_vector_type(8), aligned(2)));
typedef _Float16 h4u __attribute__((ext_vector_type(4), aligned(2)));

// p[0..W-1], elements at and past `lim` zero
template <int W, class V>
__device__ __forceinline__ V load_lim(const _Float16 * p, int lim)
{
  if (lim >= W) {
    if constexpr (W == 8) return (V)*reinterpret_cast<const h8u *>(p);
    else return (V)*reinterpret_cast<const h4u *>(p);
  }
  V v = V{};
#pragma unroll
  for (int e = 0; e < W; ++e)
    if (e < lim) v[e] = p[e];
  return v;
}

// One operand tile of R rows x kBK: registers of a K step, and their way into LDS.
// T: stored [K][rows] (row stride `rows` elements), else [rows][K].
template <int R, bool T> struct Tile {
  static constexpr int W = R == 128 ? 8 : 4;         // T: columns of a thread's 4-deep block
  static constexpr int N = T ? 4 : R / 32;           // register pieces
  typedef _Float16 vt __attribute__((ext_vector_type(T ? W : 8)));
  vt v[N];
  __device__ __forceinline__ void load(const _Float16 * p, int r0, int rows, int k0, int K)
  {
    const int tid = threadIdx.x;
    if constexpr (T) {
      const int r = r0 + ((tid >> 6) * 4 + (tid & 3)) * W, k = k0 + ((tid >> 2) & 15) * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        v[j] = k + j < K ? load_lim<W, vt>(p + (long)(k + j) * rows + r, rows - r) : vt{};
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int e = tid + 256 * i, r = r0 + (e >> 3), k = k0 + (e & 7) * 8;
        v[i] = r < rows ? load_lim<8, vt>(p + (long)r * K + k, K - k) : vt{};
      }
    }
  }
  __device__ __forceinline__ void store(_Float16 * lds) const
  {
    const int tid = threadIdx.x;
    if constexpr (T) {
      // lanes: 16 k runs x 4 column blocks, so the 8-byte writes of a wave cover every bank
      const int r = ((tid >> 6) * 4 + (tid & 3)) * W, k = ((tid >> 2) & 15) * 4;
#pragma unroll
      for (int e = 0; e < W; ++e) *reinterpret_cast<h4 *>(lds + (r + e) * kLDK + k) = h4{v[0][e], v[1][e], v[2][e], v[3][e]};
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const int e = tid + 256 * i;
        *reinterpret_cast<vt *>(lds + (e >> 3) * kLDK + (e & 7) * 8) = v[i];
      }
    }
  }
};
}  // namespace

template <int TA, int TB, int BM, int BN>
__global__ void __launch_bounds__(256) bmm_mfma_kernel(const SmallParams q, int mt, int nt)
{
  using F = Mf<32>;
  constexpr int WM = BM / 32, LDY = BN + 8;
  static_assert(WM * (BN / 64) == 4, "four waves of 32 x 64");
  static_assert(BM * LDY <= (BM + BN) * kLDK, "the output tile fits the operand tiles");
  __shared__ __attribute__((aligned(16))) _Float16 lds[(BM + BN) * kLDK];
  _Float16 * const As = lds, * const Bs = lds + BM * kLDK;
  const int BB = q.i0, M = q.i1, K = q.i2, N = q.i3;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave % WM, wn = wave / WM;
  const int lin = xcd_tile(blockIdx.x, gridDim.x), z = lin / (mt * nt), t = lin - z * (mt * nt);
  const int img = z / BB, hb = z - img * BB;
  const int m0 = t / nt * BM, n0 = t % nt * BN;
  const _Float16 * A = reinterpret_cast<const _Float16 *>(q.a.ptr) + (long)img * q.a.img + (long)hb * M * K;
  const _Float16 * B = reinterpret_cast<const _Float16 *>(q.b.ptr) + (long)img * q.b.img + (long)hb * K * N;
  _Float16 * Y = reinterpret_cast<_Float16 *>(q.y.ptr) + (long)img * q.y.img + (long)hb * M * N;

  F::acc_t acc[2];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int v = 0; v < F::NV; ++v) acc[j][v] = 0.0f;

  Tile<BM, TA != 0> ta;
  Tile<BN, TB == 0> tb;
  ta.load(A, m0, M, 0, K);
  tb.load(B, n0, N, 0, K);
  for (int k0 = 0; k0 < K; k0 += kBK) {
    if (k0) __syncthreads();  // the previous step's fragments are read
    ta.store(As);
    tb.store(Bs);
    __syncthreads();
    if (k0 + kBK < K) {
      ta.load(A, m0, M, k0 + kBK, K);
      tb.load(B, n0, N, k0 + kBK, K);
    }
#pragma unroll
    for (int j = 0; j < kBK / 16; ++j) {
      const h8 fa = *reinterpret_cast<const h8 *>(As + (wm * 32 + (lane & 31)) * kLDK + j * 16 + F::kq(lane));
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const h8 fb = *reinterpret_cast<const h8 *>(Bs + (wn * 64 + u * 32 + (lane & 31)) * kLDK + j * 16 + F::kq(lane));
        acc[u] = F::mma(fb, fa, acc[u]);
      }
    }
  }
  __syncthreads();
  // D: lane holds row m = lane % 32 of the wave's rows, runs of four columns n
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int v4 = 0; v4 < F::NV; v4 += 4)
      *reinterpret_cast<h4 *>(lds + (wm * 32 + (lane & 31)) * LDY + wn * 64 + u * 32 + F::row(lane, v4)) =
          h4{(_Float16)acc[u][v4], (_Float16)acc[u][v4 + 1], (_Float16)acc[u][v4 + 2], (_Float16)acc[u][v4 + 3]};
  __syncthreads();
  constexpr int PR = BN / 8;  // pieces per row
#pragma unroll
  for (int i = 0; i < BM * PR / 256; ++i) {
    const int e = tid + 256 * i, r = e / PR, n8 = e % PR * 8, m = m0 + r, n = n0 + n8;
    if (m >= M || n >= N) continue;
    const h8 v = *reinterpret_cast<const h8 *>(lds + r * LDY + n8);
    _Float16 * yp = Y + (long)m * N + n;
    if (n + 8 <= N) *reinterpret_cast<h8u *>(yp) = (h8u)v;
    else
      for (int c = 0; c < 8 && n + c < N; ++c) yp[c] = v[c];
  }
}

// Tile rows and columns: up to 64 columns a tile of 128 would be half empty.
static long tiles(const SmallParams & q, long & mt, long & nt)
{
  const long bm = q.i3 <= 64 ? 128 : 64, bn = q.i3 <= 64 ? 64 : 128;
  mt = (q.i1 + bm - 1) / bm;
  nt = (q.i3 + bn - 1) / bn;
  return mt * nt;
}

template <int TA, int TB>
static void launch_bmm_t(const SmallParams & q, hipStream_t s)
{
  long mt, nt;
  const long n = tiles(q, mt, nt) * q.batch * q.i0;
  const dim3 grid((unsigned)n), block(256);
  if (q.i3 <= 64) hipLaunchKernelGGL((bmm_mfma_kernel<TA, TB, 128, 64>), grid, block, 0, s, q, (int)mt, (int)nt);
  else hipLaunchKernelGGL((bmm_mfma_kernel<TA, TB, 64, 128>), grid, block, 0, s, q, (int)mt, (int)nt);
}

// q.op bit 0: A stored [K][M]; bit 1: B stored [N][K].  A launch holds fewer than 2^32 lanes per
// grid dimension, 2^24 work-groups here: more tiles are launched as slices of the images, or of
// one image's matrices.
void launch_bmm_mfma(const SmallParams & q, hipStream_t s)
{
  constexpr long kMaxWgs = (1L << 24) - 1;
  long mt, nt;
  const long per = tiles(q, mt, nt);
  if (per > kMaxWgs) {  // a matrix of one row or column of nearly 2^31 values (K = 1): in two parts
    if (q.i0 != 1 || q.i2 != 1) throw std::runtime_error("bmm grid");
    SmallParams c = q;
    const bool rows = q.i1 > q.i3;
    int & d = rows ? c.i1 : c.i3;
    const int part = 1 << 30, all = d;
    d = part;
    launch_bmm_mfma(c, s);
    (rows ? c.a : c.b).ptr += part;
    c.y.ptr += part;
    d = all - part;
    launch_bmm_mfma(c, s);
    return;
  }
  if (per * q.i0 > kMaxWgs || per * q.i0 * q.batch > kMaxWgs) {
    const bool heads = per * q.i0 > kMaxWgs;
    const int step = (int)(kMaxWgs / (heads ? per : per * q.i0)), all = heads ? q.i0 : q.batch;
    for (int img = 0; img < (heads ? q.batch : 1); ++img)
      for (int at = 0; at < all; at += step) {
        SmallParams c = q;
        (heads ? c.i0 : c.batch) = std::min(step, all - at);
        if (heads) c.batch = 1;
        const long i = heads ? img : at, h = heads ? at : 0;
        c.a.ptr += i * q.a.img + h * q.i1 * q.i2;
        c.b.ptr += i * q.b.img + h * q.i2 * q.i3;
        c.y.ptr += i * q.y.img + h * q.i1 * q.i3;
        launch_bmm_mfma(c, s);
      }
    return;
  }
  switch (q.op & 3) {
  case 0: launch_bmm_t<0, 0>(q, s); break;
  case 1: launch_bmm_t<1, 0>(q, s); break;
  case 2: launch_bmm_t<0, 1>(q, s); break;
  default: launch_bmm_t<1, 1>(q, s); break;
  }
}

}  // namespace ivh
