// unet_kernels.hip -- kernels of the learned WFF2 surrogate (a 4-level U-Net)
// on gfx950: 3x3 convolutions as implicit GEMMs on BF16 MFMA
// (v_mfma_f32_16x16x32_bf16, FP32 accumulation) for the forward pass, the
// input gradient and the weight gradient, plus the small VALU kernels around
// them (2-channel input layer, 1x1 output layer with the loss, max pooling,
// upsampling adjoint, Adam).
//
// Layouts: activations NHWC bf16 (channels innermost, counts multiples of 32
// except the 2-channel input/output); weights [Cout][9][Cin] bf16 for the
// forward pass (K = tap*Cin + ci contiguous per output channel) and
// [Cin][9][Cout] with flipped taps for the input gradient; FP32 master
// weights, gradients and Adam moments in the [Cout][3][3][Cin] order.
#include "unet_internal.h"

#include <algorithm>
#include <atomic>

namespace glsu {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

__device__ __forceinline__ bf16x8 zero8() {
  bf16x8 z;
#pragma unroll
  for (int i = 0; i < 8; ++i) z[i] = (__bf16)0.f;
  return z;
}

// 8 channels [c, c+8) of pixel (n, y, x) of the (virtual) concatenation
// cat(X1, up2(X2)); zero outside the image.  c is a multiple of 8 and a
// 32-channel chunk never straddles the two sources (C1 % 32 == 0).
__device__ __forceinline__ bf16x8 load8(const __bf16* __restrict__ X1, int C1,
                                        const __bf16* __restrict__ X2, int C2, int n, int y,
                                        int x, int H, int W, int c) {
  if (y < 0 || y >= H || x < 0 || x >= W) return zero8();
  if (c < C1) return *(const bf16x8*)(X1 + (((size_t)n * H + y) * W + x) * C1 + c);
  const int H2 = H >> 1, W2 = W >> 1;
  return *(const bf16x8*)(X2 + (((size_t)n * H2 + (y >> 1)) * W2 + (x >> 1)) * C2 + (c - C1));
}

// The same value as load8 without a branch around the load: the pixel is
// clamped into the image, loaded unconditionally and replaced by zero when it
// was outside, so that a thread's loads can all be in flight together.
__device__ __forceinline__ bf16x8 load8_clamped(const __bf16* __restrict__ X1, int C1,
                                                const __bf16* __restrict__ X2, int C2, int n,
                                                int y, int x, int H, int W, int c) {
  const bool in = y >= 0 && y < H && x >= 0 && x < W;
  const int yc = min(max(y, 0), H - 1), xc = min(max(x, 0), W - 1);
  bf16x8 v;
  if (c < C1) {
    v = *(const bf16x8*)(X1 + (((size_t)n * H + yc) * W + xc) * C1 + c);
  } else {
    const int H2 = H >> 1, W2 = W >> 1;
    v = *(const bf16x8*)(X2 + (((size_t)n * H2 + (yc >> 1)) * W2 + (xc >> 1)) * C2 + (c - C1));
  }
  return in ? v : zero8();
}

// ------------------------------------------------------------------------
// 3x3 convolution, implicit GEMM over pixels x output channels, K = 9*Cin.
// Workgroup: 4 waves, output tile 4 rows x 64 pixels x NCO channels; wave w
// owns row w.  Per 32-channel chunk the input tile (6 x 66 pixels x 32
// channels, 25 KB) is staged in LDS; each 16-byte group of 8 channels of LDS
// pixel p sits at group slot g ^ ((p >> 1) & 3), which keeps the MFMA operand
// reads (16 consecutive pixels, one group) free of bank conflicts without
// padding.  Weights: 32-channel tiles read them straight from global memory
// (small and shared by every workgroup, so they stay in L1/L2), one tap ahead
// of their use; 64-channel tiles stage them in LDS one row of three taps at a
// time.  The weights are the MFMA A operand and the pixels the B operand, so
// a lane's accumulators hold four consecutive output channels of one pixel.
// Each wave issues 4 x (NCO/16) MFMAs per tap.
// MODE 0: y = relu(acc + bias).  MODE 1: y = acc * (mask > 0) (mask may be
// null: y = acc).  Used for the forward pass (weights [Cout][9][Cin]) and
// for the input gradient (dY as input, flipped transposed weights).
// LDS rows of the staged tile are kInPitch = 72 pixels apart (a multiple of
// 8), so the bank swizzle of a fragment depends only on the lane and dx: the
// fragment reads are immediate offsets from three per-lane bases, and the
// staging slots, their LDS offsets and (away from the image border) their
// global offsets are per-thread constants.
constexpr int kTileW = 64, kTileH = 4;
constexpr int kInW = kTileW + 2, kInPitch = kTileW + 8;
constexpr int kInSlots = (kTileH + 2) * kInPitch * 4;  // 16-byte slots of the staged tile

__device__ __forceinline__ int swz(int p, int g) { return p * 32 + ((g ^ ((p >> 1) & 3)) << 3); }
// byte offset of 16-byte group g of LDS pixel p (the same swizzle)
__device__ __forceinline__ int swz_b(int p, int g) { return p * 64 + ((g ^ ((p >> 1) & 3)) << 4); }

template <int NCO, int MODE>
__global__ __launch_bounds__(256) void conv3_mfma_kernel(
    const __bf16* __restrict__ X1, int C1, const __bf16* __restrict__ X2, int C2,
    const __bf16* __restrict__ Wt, const float* __restrict__ bias,
    const __bf16* __restrict__ mask, __bf16* __restrict__ Y, int n, int H, int W, int Cout) {
  constexpr int NB = NCO / 16;
  // 64-channel tiles read each weight fragment from 4 waves: stage the weights
  // in LDS, one row of 3 taps at a time; 32-channel tiles read them from
  // global memory (L1), which leaves LDS for more resident workgroups
  constexpr bool kWLds = NCO >= 64;
  __shared__ __attribute__((aligned(16))) char sIn[kInSlots * 16];
  __shared__ __attribute__((aligned(16))) char sW[kWLds ? 3 * NCO * 64 : 16];
  const int Cin = C1 + C2;
  const int tilesx = (W + kTileW - 1) / kTileW;
  const int tilesy = H / kTileH;
  const int tile = blockIdx.x;
  const int img = tile / (tilesx * tilesy);
  const int ty = (tile / tilesx) % tilesy, tx = tile % tilesx;
  const int y0 = ty * kTileH, x0 = tx * kTileW;
  const int co0 = blockIdx.y * NCO;
  const int tid = threadIdx.x;
  const int wave = tid / 64, lane = tid % 64;
  const int lr = lane % 16, lk = lane / 16;

  // staging slot r of this thread: LDS pixel sp = tid/4 + 64 r, group sg =
  // tid % 4, at byte sbase + 4096 r (the swizzle term of sp is (tid >> 3) & 3
  // for every r); live bit r: the slot is a tile pixel, not row padding
  constexpr int kLd = (kInSlots + 255) / 256;
  const int sg = tid & 3;
  const int sbase = swz_b(tid >> 2, sg);
  const bool interior = y0 >= 1 && y0 + kTileH + 1 <= H && x0 >= 1 && x0 + kTileW + 1 <= W;
  unsigned live = 0;
  int off1[kLd];  // X1 element offset from the tile's corner (interior tiles)
#pragma unroll
  for (int r = 0; r < kLd; ++r) {
    const int sp = (tid >> 2) + 64 * r, ry = sp / kInPitch, rx = sp % kInPitch;
    live |= (sp < kInSlots / 4 && rx < kInW ? 1u : 0u) << r;
    off1[r] = (ry * W + rx) * C1 + sg * 8;
  }
  // fragment bases: pixel (wave + dy, 16 mb + lr + dx) of the tile sits at
  // pbase[dx] + (dy * kInPitch + 16 mb) * 64
  int pbase[3];
#pragma unroll
  for (int dx = 0; dx < 3; ++dx) pbase[dx] = swz_b(wave * kInPitch + lr + dx, lk);

  floatx4 acc[4][NB];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  // weight operand of block nb at tap t of chunk ci0: channel co0 + 16 nb + lr,
  // input channels ci0 + 8 lk .. + 7
  auto load_b = [&](bf16x8* b, int t, int ci0) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int co = co0 + nb * 16 + lr;
      b[nb] = co < Cout ? *(const bf16x8*)(Wt + ((size_t)co * 9 + t) * Cin + ci0 + lk * 8)
                        : zero8();
    }
  };
  auto tap = [&](int t, const bf16x8* b) {
    const int dy = t / 3, dx = t % 3;  // offsets + 1
    bf16x8 a[4];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
      a[mb] = *(const bf16x8*)(sIn + pbase[dx] + (dy * kInPitch + mb * 16) * 64);
    // weights as the A operand, pixels as B: the 16 x 16 result is
    // [output channel][pixel], so each lane ends with 4 consecutive channels
    // of one pixel (one 8-byte NHWC store in the epilogue)
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[nb], a[mb], acc[mb][nb], 0, 0, 0);
  };

  // weight staging (NCO >= 64): one row of three taps, 3 * NCO * 32 bf16, as
  // kWl 16-byte loads per thread, all issued before any is stored; the next
  // row's loads are in flight during the current row's MFMAs
  // weight slot r (tap tl of the row, channel co = sp / NCO, sp % NCO) at the
  // same LDS offsets as the tile's slots; its global offset less 3 tg Cin + ci0
  constexpr int kWl = (3 * NCO * 4 + 255) / 256;
  bf16x8 wl[kWLds ? kWl : 1];
  int offw[kWLds ? kWl : 1];
  unsigned wlive = 0;
  if constexpr (kWLds) {
#pragma unroll
    for (int r = 0; r < kWl; ++r) {
      const int sp = (tid >> 2) + 64 * r, tl = min(sp / NCO, 2), co = sp % NCO;
      wlive |= (sp < 3 * NCO && co0 + co < Cout ? 1u : 0u) << r;
      offw[r] = (min(co0 + co, Cout - 1) * 9 + tl) * Cin + sg * 8;
    }
  }
  const int wbase = swz_b(lr, lk);
  auto load_w = [&](int tg, int ci0) {
#pragma unroll
    for (int r = 0; r < kWl; ++r) {
      const bf16x8 v = *(const bf16x8*)(Wt + offw[r] + 3 * tg * Cin + ci0);
      wl[r] = (wlive >> r) & 1 ? v : zero8();
    }
  };
  auto store_w = [&]() {
#pragma unroll
    for (int r = 0; r < kWl; ++r)
      if ((tid >> 2) + 64 * r < 3 * NCO) *(bf16x8*)(sW + sbase + 4096 * r) = wl[r];
  };

  for (int ci0 = 0; ci0 < Cin; ci0 += 32) {
    bf16x8 b[NB];
    if (!kWLds) load_b(b, 0, ci0);
    if constexpr (kWLds) load_w(0, ci0);
    // the chunk's input tile: every 16-byte load of this thread is issued
    // before the first is stored (one memory round trip, not one per load)
    bf16x8 ld[kLd];
    if (interior && ci0 < C1) {
      const __bf16* base = X1 + (((size_t)img * H + (y0 - 1)) * W + (x0 - 1)) * C1 + ci0;
#pragma unroll
      for (int r = 0; r < kLd; ++r) ld[r] = *(const bf16x8*)(base + off1[r]);
    } else {
#pragma unroll
      for (int r = 0; r < kLd; ++r) {
        const int sp = min((tid >> 2) + 64 * r, kInSlots / 4 - 1);
        const int ry = sp / kInPitch, rx = min(sp % kInPitch, kInW - 1);
        ld[r] = load8_clamped(X1, C1, X2, C2, img, y0 + ry - 1, x0 + rx - 1, H, W, ci0 + sg * 8);
      }
    }
    __syncthreads();  // previous chunk fully consumed
#pragma unroll
    for (int r = 0; r < kLd; ++r)
      if ((live >> r) & 1) *(bf16x8*)(sIn + sbase + 4096 * r) = ld[r];
    if constexpr (kWLds) {
#pragma unroll
      for (int tg = 0; tg < 3; ++tg) {
        if (tg > 0) __syncthreads();  // previous tap row consumed
        store_w();
        if (tg < 2) load_w(tg + 1, ci0);
        __syncthreads();
#pragma unroll
        for (int tl = 0; tl < 3; ++tl) {
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
            b[nb] = *(const bf16x8*)(sW + wbase + (tl * NCO + nb * 16) * 64);
          tap(3 * tg + tl, b);
        }
      }
    } else {
      __syncthreads();
#pragma unroll 1
      for (int t = 0; t < 9; ++t) {
        bf16x8 bn[NB];
        if (t < 8) load_b(bn, t + 1, ci0);
        tap(t, b);
        if (t < 8) {
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) b[nb] = bn[nb];
        }
      }
    }
  }
  // epilogue: lane holds rows 4*lk + j (output channels) of column lr (pixel)
  const int y = y0 + wave;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int cb = co0 + nb * 16 + 4 * lk;  // channels cb .. cb + 3 (Cout % 16 == 0)
    if (cb >= Cout) continue;
    float bv[4] = {0.f, 0.f, 0.f, 0.f};
    if (MODE == 0)
#pragma unroll
      for (int j = 0; j < 4; ++j) bv[j] = bias[cb + j];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      const int x = x0 + mb * 16 + lr;
      if (x >= W) continue;
      const size_t o = (((size_t)img * H + y) * W + x) * Cout + cb;
      bf16x4 out;
      bf16x4 mk;
      if (MODE == 1 && mask) mk = *(const bf16x4*)(mask + o);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float v = acc[mb][nb][j];
        if (MODE == 0) {
          v = fmaxf(v + bv[j], 0.f);
        } else if (mask) {
          v = ((float)mk[j] > 0.f) ? v : 0.f;
        }
        out[j] = (__bf16)v;
      }
      *(bf16x4*)(Y + o) = out;
    }
  }
}

// ------------------------------------------------------------------------
// 3x3 convolution, the same implicit GEMM, persistent and software-pipelined,
// with its addressing reduced to per-thread constants (the kernel above spends
// more issue cycles on address arithmetic than on MFMAs).  Used for 32 output
// channels (the full-resolution layers); with 64-channel tiles the per-item
// restaging of 9 x 64 x 32 weights made it slower than the kernel above.
// Workgroup: 4 waves in a 2 x 2 grid, output tile 8 rows x 32 PX pixels x NCO
// channels (NCO = 32: PX = 2); wave (wr, wc) owns rows
// 4 wr .. 4 wr + 3 and pixels 16 PX wc .. + 16 PX - 1.  The workgroup runs the
// items (tile, 32-channel chunk) of tiles b, b + G, ... (G workgroups); the
// next item's input tile (10 x (32 PX + 2) pixels) and weights (9 x NCO x 32,
// loaded once when there is a single chunk) are read into registers while the
// current item's MFMAs run and stored to LDS after them, two barriers per
// item.  LDS rows are 32 PX + 8 pixels apart (a multiple of 8), so the bank
// swizzle of a fragment depends only on the lane and dx and every fragment
// read is an immediate offset from one of three per-lane bases; staging slots
// and their global offsets are per-thread constants, and tiles away from the
// image border load without clamping.  The taps run by column dx: each of the
// wave's 6 input rows is read once per dx (PX 16-pixel fragments) and applied
// to every output row that uses it (dy = input row - output row).
// Same modes and results (up to the FP32 summation order) as the kernel above.
constexpr int kRTileH = 8, kRInRows = kRTileH + 2;
template <int NCO>
struct RowsConv {
  static constexpr int PX = NCO == 32 ? 2 : 1;       // 16-pixel blocks per wave row
  static constexpr int Q = NCO / 16;                 // 16-channel blocks
  static constexpr int TW = 32 * PX;                 // tile width (pixels)
  static constexpr int InW = TW + 2;                 // staged pixels per row
  static constexpr int Pitch = TW + 8;               // LDS pixels per tile row
  static constexpr int Slots = kRInRows * Pitch * 4; // 16-byte LDS slots of the tile
  static constexpr int Ld = (Slots + 255) / 256;     // per thread
  static constexpr int WSlots = 9 * NCO * 4;         // weight slots (taps x co x groups)
  static constexpr int Wl = (WSlots + 255) / 256;
};

// 2 x 2 max-pool of a ReLU conv output still held as MFMA accumulators: rows
// o and o + 1 are two registers of the lane (a, b), pixels x and x + 1 two
// adjacent lanes (lr even / odd).  Every value is rounded to bf16 before the
// maximum, so the result equals maxpool2_kernel's on the stored output.  All
// 64 lanes must call it (lane exchange); the even lanes hold the result.
__device__ __forceinline__ bf16x4 pool_pair(const floatx4& a, const floatx4& b,
                                            const float (&bv)[4]) {
  bf16x4 r;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float u = (float)(__bf16)fmaxf(a[j] + bv[j], 0.f);
    const float v = (float)(__bf16)fmaxf(b[j] + bv[j], 0.f);
    float m = fmaxf(u, v);
    m = fmaxf(m, __shfl_xor(m, 1));
    r[j] = (__bf16)m;
  }
  return r;
}

template <int NCO, int MODE>
__global__ __launch_bounds__(256, 2) void conv3_rows_kernel(
    const __bf16* __restrict__ X1, int C1, const __bf16* __restrict__ X2, int C2,
    const __bf16* __restrict__ Wt, const float* __restrict__ bias,
    const __bf16* __restrict__ mask, __bf16* __restrict__ Y, int n, int H, int W, int Cout,
    __bf16* __restrict__ pool) {
  static_assert(NCO == 32, "64-channel tiles use conv3_res64_kernel or conv3_mfma_kernel");
  using K = RowsConv<NCO>;
  constexpr int Q = K::Q, P = K::PX, R = 4;
  constexpr int kRTileW = K::TW, kRInW = K::InW, kRPitch = K::Pitch;
  constexpr int kRLd = K::Ld, kRWl = K::Wl;
  __shared__ __attribute__((aligned(16))) char sIn[kRInRows * kRPitch * 64];
  __shared__ __attribute__((aligned(16))) char sW[K::WSlots * 16];
  const int Cin = C1 + C2;
  const bool one_chunk = Cin == 32;
  const int tilesx = (W + kRTileW - 1) / kRTileW;
  const int tilesy = H / kRTileH;
  const int ntiles = n * tilesy * tilesx;
  const int co0 = blockIdx.y * NCO;
  const int tid = threadIdx.x;
  const int wave = tid / 64, lane = tid % 64;
  const int wr = wave / 2, wc = wave % 2;
  const int lr = lane % 16, lk = lane / 16;

  // staging slot r of this thread: LDS pixel sp = tid/4 + 64 r, group sg =
  // tid % 4; its LDS byte offset is sbase + 4096 r (the swizzle term of sp is
  // (tid >> 3) & 3 for every r)
  const int sg = tid & 3;
  const int sbase = swz_b(tid >> 2, sg);
  unsigned live = 0;   // bit r: slot r is a tile pixel (not row padding / past the end)
  int off1[kRLd];      // X1 element offset from the item's corner (interior tiles)
#pragma unroll
  for (int r = 0; r < kRLd; ++r) {
    const int sp = (tid >> 2) + 64 * r, ry = sp / kRPitch, rx = sp % kRPitch;
    const bool ok = sp < kRInRows * kRPitch && rx < kRInW;
    live |= (ok ? 1u : 0u) << r;
    off1[r] = (ry * W + rx) * C1 + sg * 8;
  }
  // weight slot r: (tap t, channel co) = sp / 32, sp % 32 at the same LDS offsets
  int offw[kRWl];
  unsigned wlive = 0;
#pragma unroll
  for (int r = 0; r < kRWl; ++r) {
    const int sp = (tid >> 2) + 64 * r, t = sp / NCO, co = sp % NCO;
    const bool ok = sp < 9 * NCO && co0 + co < Cout;
    wlive |= (ok ? 1u : 0u) << r;
    offw[r] = ((min(co0 + co, Cout - 1) * 9 + min(t, 8)) * Cin) + sg * 8;
  }

  bf16x8 ld[kRLd], wl[kRWl];
  auto load_w = [&](int ci0) {
#pragma unroll
    for (int r = 0; r < kRWl; ++r) {
      const bf16x8 v = *(const bf16x8*)(Wt + offw[r] + ci0);
      wl[r] = (wlive >> r) & 1 ? v : zero8();
    }
  };
  auto load_item = [&](int tile, int ci0, bool with_w) {
    const int img = tile / (tilesx * tilesy);
    const int y0 = ((tile / tilesx) % tilesy) * kRTileH, x0 = (tile % tilesx) * kRTileW;
    const bool interior = y0 >= 1 && y0 + kRTileH + 1 <= H && x0 >= 1 && x0 + kRTileW + 1 <= W;
    if (interior && ci0 < C1) {
      const __bf16* base = X1 + (((size_t)img * H + (y0 - 1)) * W + (x0 - 1)) * C1 + ci0;
#pragma unroll
      for (int r = 0; r < kRLd; ++r) ld[r] = *(const bf16x8*)(base + off1[r]);
    } else {
#pragma unroll
      for (int r = 0; r < kRLd; ++r) {
        const int sp = min((tid >> 2) + 64 * r, kRInRows * kRPitch - 1);
        const int ry = sp / kRPitch, rx = min(sp % kRPitch, kRInW - 1);
        ld[r] = load8_clamped(X1, C1, X2, C2, img, y0 + ry - 1, x0 + rx - 1, H, W, ci0 + sg * 8);
      }
    }
    if (with_w) load_w(ci0);
  };
  auto store_item = [&](bool with_w) {
#pragma unroll
    for (int r = 0; r < kRLd; ++r)
      if ((live >> r) & 1) *(bf16x8*)(sIn + sbase + 4096 * r) = ld[r];
    if (with_w) {
#pragma unroll
      for (int r = 0; r < kRWl; ++r)
        if ((tid >> 2) + 64 * r < 9 * NCO) *(bf16x8*)(sW + sbase + 4096 * r) = wl[r];
    }
  };

  // fragment bases: pixel (4 wr + r, 16 P wc + 16 p + lr + dx) of the tile sits at
  // pbase[dx] + (r * kRPitch + 16 p) * 64; weight (tap t, 16 q + lr) at
  // wbase + (t * NCO + 16 q) * 64
  int pbase[3];
#pragma unroll
  for (int dx = 0; dx < 3; ++dx)
    pbase[dx] = swz_b(4 * wr * kRPitch + 16 * P * wc + lr + dx, lk);
  const int wbase = swz_b(lr, lk);

  int tile = blockIdx.x;  // uniform per workgroup: every barrier below is reached by all waves
  if (tile >= ntiles) return;
  load_item(tile, 0, true);
  bool first = true;
  for (; tile < ntiles; tile += gridDim.x) {
    floatx4 acc[R][P][Q];
#pragma unroll
    for (int o = 0; o < R; ++o)
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[o][p][q] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int ci0 = 0; ci0 < Cin; ci0 += 32) {
      const bool w_now = first || !one_chunk;
      __syncthreads();  // the previous item's LDS reads are done
      store_item(w_now);
      __syncthreads();
      first = false;
      {  // the next item's loads, in flight during this item's MFMAs
        int nt = tile, nc = ci0 + 32;
        if (nc >= Cin) {
          nt = tile + gridDim.x;
          nc = 0;
        }
        if (nt < ntiles) load_item(nt, nc, !one_chunk);
      }
#pragma unroll
      for (int dx = 0; dx < 3; ++dx) {
        // weights as the A operand, pixels as B (lane: 4 channels of one pixel)
        bf16x8 wf[3][Q];
#pragma unroll
        for (int dy = 0; dy < 3; ++dy)
#pragma unroll
          for (int q = 0; q < Q; ++q)
            wf[dy][q] = *(const bf16x8*)(sW + wbase + ((3 * dy + dx) * NCO + 16 * q) * 64);
#pragma unroll
        for (int r = 0; r < R + 2; ++r) {  // input row 4 wr + r of the tile
          bf16x8 pf[P];
#pragma unroll
          for (int p = 0; p < P; ++p)
            pf[p] = *(const bf16x8*)(sIn + pbase[dx] + (r * kRPitch + 16 * p) * 64);
#pragma unroll
          for (int o = 0; o < R; ++o) {
            const int dy = r - o;
            if (dy < 0 || dy > 2) continue;
#pragma unroll
            for (int p = 0; p < P; ++p)
#pragma unroll
              for (int q = 0; q < Q; ++q)
                acc[o][p][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[dy][q], pf[p],
                                                                       acc[o][p][q], 0, 0, 0);
          }
        }
      }
    }
    // epilogue: lane holds channels 4 lk .. 4 lk + 3 of block q, pixel lr of block p
    const int img = tile / (tilesx * tilesy);
    const int y0 = ((tile / tilesx) % tilesy) * kRTileH, x0 = (tile % tilesx) * kRTileW;
    const bool full = x0 + kRTileW <= W && co0 + NCO <= Cout;
    const size_t tbase = (((size_t)img * H + y0 + 4 * wr) * W + x0 + 16 * P * wc) * Cout + co0;
    float bv[Q][4];  // read per tile: kept out of the registers of the MFMA loop
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        bv[q][j] = MODE == 0 ? bias[min(co0 + q * 16 + 4 * lk + j, Cout - 1)] : 0.f;
#pragma unroll
    for (int o = 0; o < R; ++o) {
      __bf16* yrow = Y + tbase + (size_t)o * W * Cout;
      const __bf16* mrow = MODE == 1 && mask ? mask + tbase + (size_t)o * W * Cout : nullptr;
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          const int lo = (16 * p + lr) * Cout + 16 * q + 4 * lk;
          if (!full && (x0 + 16 * P * wc + 16 * p + lr >= W || co0 + 16 * q + 4 * lk >= Cout))
            continue;
          bf16x4 out;
          bf16x4 mk;
          if (MODE == 1 && mask) mk = *(const bf16x4*)(mrow + lo);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            float v = acc[o][p][q][j];
            if (MODE == 0) {
              v = fmaxf(v + bv[q][j], 0.f);
            } else if (mask) {
              v = ((float)mk[j] > 0.f) ? v : 0.f;
            }
            out[j] = (__bf16)v;
          }
          *(bf16x4*)(yrow + lo) = out;
        }
    }
    if constexpr (MODE == 0) {
      if (pool) {  // fused 2 x 2 max-pool (H, W even; rows y0 + 4 wr + o, o even, pair up)
        const int H2 = H >> 1, W2 = W >> 1;
#pragma unroll
        for (int o = 0; o < R; o += 2) {
          const int y2 = (y0 + 4 * wr + o) >> 1;
#pragma unroll
          for (int p = 0; p < P; ++p) {
            const int x = x0 + 16 * P * wc + 16 * p + lr;
#pragma unroll
            for (int q = 0; q < Q; ++q) {
              const int cb = co0 + 16 * q + 4 * lk;
              const bf16x4 m = pool_pair(acc[o][p][q], acc[o + 1][p][q], bv[q]);
              if (!(lr & 1) && x < W && cb < Cout)
                *(bf16x4*)(pool + (((size_t)img * H2 + y2) * W2 + (x >> 1)) * Cout + cb) = m;
            }
          }
        }
      }
    }
  }
}

// ------------------------------------------------------------------------
// 3x3 convolution for 64 output channels with the workgroup's weights in LDS.
// Up to 64 input channels (STREAM = false) every weight of the workgroup's 64
// output channels stays resident for the whole kernel (9 x 64 x Cin bf16,
// loaded once), so that the per-tile work is the input tile only; above that
// (STREAM = true) LDS holds one 32-channel chunk of weights, loaded into
// registers together with the input tile of the next item and stored after the
// same barrier.  Workgroup: 8 waves, 4 x 2 grid, output tile 16 rows x 32
// pixels x 64 channels; wave (wr, wc) owns rows 4 wr .. 4 wr + 3 and pixels
// 16 wc .. 16 wc + 15.  Persistent over items (tile, 32-channel chunk) like
// conv3_rows_kernel, the next item's 18 x 34-pixel tile loaded into registers
// during the current item's MFMAs; LDS rows 40 pixels apart, so fragment reads
// are immediate offsets from per-lane bases.  One workgroup per CU (83-120 KB
// of LDS), two waves per SIMD.  Same modes and results (up to the FP32
// summation order) as conv3_mfma_kernel.
constexpr int kXTileH = 16, kXTileW = 32, kXInRows = kXTileH + 2, kXInW = kXTileW + 2,
              kXPitch = kXTileW + 8;
constexpr int kXSlots = kXInRows * kXPitch * 4;  // 16-byte slots of the tile
constexpr int kXLd = (kXSlots + 511) / 512;       // per thread
constexpr int kXMaxCin = 64;
constexpr int kXWLd = (9 * 64 * 4 + 511) / 512;   // weight slots of one chunk per thread

template <int MODE, bool STREAM>
__global__ __launch_bounds__(512, 1) void conv3_res64_kernel(
    const __bf16* __restrict__ X1, int C1, const __bf16* __restrict__ X2, int C2,
    const __bf16* __restrict__ Wt, const float* __restrict__ bias,
    const __bf16* __restrict__ mask, __bf16* __restrict__ Y, int n, int H, int W, int Cout,
    __bf16* __restrict__ pool) {
  constexpr int NCO = 64, Q = 4, R = 4;
  __shared__ __attribute__((aligned(16))) char sIn[kXInRows * kXPitch * 64];
  __shared__ __attribute__((aligned(16))) char sW[(STREAM ? 1 : kXMaxCin / 32) * 9 * NCO * 64];
  const int Cin = C1 + C2, nch = Cin / 32;
  const int tilesx = (W + kXTileW - 1) / kXTileW;
  const int tilesy = H / kXTileH;
  const int ntiles = n * tilesy * tilesx;
  const int co0 = blockIdx.y * NCO;
  const int tid = threadIdx.x;
  const int wave = tid / 64, lane = tid % 64;
  const int wr = wave / 2, wc = wave % 2;
  const int lr = lane % 16, lk = lane / 16;
  const int sg = tid & 3;
  // staging slot r of this thread: LDS pixel tid/4 + 128 r, group sg, at byte
  // sbase + 8192 r (the swizzle term of that pixel is (tid >> 3) & 3 for every r)
  const int sbase = swz_b(tid >> 2, sg);

  // all weights of the workgroup's channels: LDS pixel (c 9 + t) NCO + co
  if constexpr (!STREAM) {
    const int nslot = nch * 9 * NCO * 4;
    for (int i = tid; i < nslot; i += 512) {
      const int g = i & 3, px = i >> 2;
      const int co = px % NCO, ct = px / NCO, c = ct / 9, t = ct % 9;
      bf16x8 v = zero8();
      if (co0 + co < Cout) v = *(const bf16x8*)(Wt + ((size_t)(co0 + co) * 9 + t) * Cin + c * 32 + g * 8);
      *(bf16x8*)(sW + swz_b(px, g)) = v;
    }
  }

  unsigned live = 0;
  int off1[kXLd];
#pragma unroll
  for (int r = 0; r < kXLd; ++r) {
    const int sp = (tid >> 2) + 128 * r, ry = sp / kXPitch, rx = sp % kXPitch;
    live |= (sp < kXInRows * kXPitch && rx < kXInW ? 1u : 0u) << r;
    off1[r] = (ry * W + rx) * C1 + sg * 8;
  }
  // STREAM: weight slot r of this thread is LDS pixel tid/4 + 128 r of the
  // chunk, i.e. tap (tid >> 8) + 2 r of output channel (tid >> 2) & 63, group
  // sg, stored at the same sbase + 8192 r as the tile's slots
  const int wco = (tid >> 2) & 63;
  const bool wok = co0 + wco < Cout;
  int woff[kXWLd];
  unsigned wlive = 0;
#pragma unroll
  for (int r = 0; r < kXWLd; ++r) {
    const int t = (tid >> 8) + 2 * r;
    wlive |= (t < 9 && wok ? 1u : 0u) << r;
    woff[r] = ((co0 + wco) * 9 + min(t, 8)) * Cin + sg * 8;
  }
  bf16x8 ld[kXLd];
  bf16x8 wl[STREAM ? kXWLd : 1];
  auto load_item = [&](int tile, int ci0) {
    if constexpr (STREAM) {
#pragma unroll
      for (int r = 0; r < kXWLd; ++r)
        wl[r] = ((wlive >> r) & 1) ? *(const bf16x8*)(Wt + woff[r] + ci0) : zero8();
    }
    const int img = tile / (tilesx * tilesy);
    const int y0 = ((tile / tilesx) % tilesy) * kXTileH, x0 = (tile % tilesx) * kXTileW;
    const bool interior = y0 >= 1 && y0 + kXTileH + 1 <= H && x0 >= 1 && x0 + kXTileW + 1 <= W;
    if (interior && ci0 < C1) {
      const __bf16* base = X1 + (((size_t)img * H + (y0 - 1)) * W + (x0 - 1)) * C1 + ci0;
#pragma unroll
      for (int r = 0; r < kXLd; ++r) ld[r] = *(const bf16x8*)(base + off1[r]);
    } else {
      int t2 = tid;
      __asm__ volatile("" : "+v"(t2));
#pragma unroll
      for (int r = 0; r < kXLd; ++r) {
        const int sp = min((t2 >> 2) + 128 * r, kXInRows * kXPitch - 1);
        const int ry = sp / kXPitch, rx = min(sp % kXPitch, kXInW - 1);
        ld[r] = load8_clamped(X1, C1, X2, C2, img, y0 + ry - 1, x0 + rx - 1, H, W, ci0 + sg * 8);
      }
    }
  };

  int pbase[3];
#pragma unroll
  for (int dx = 0; dx < 3; ++dx) pbase[dx] = swz_b(4 * wr * kXPitch + 16 * wc + lr + dx, lk);
  const int wbase = swz_b(lr, lk);

  int tile = blockIdx.x;  // uniform per workgroup: every barrier below is reached by all waves
  if (tile >= ntiles) return;
  load_item(tile, 0);
  for (; tile < ntiles; tile += gridDim.x) {
    floatx4 acc[R][Q];
#pragma unroll
    for (int o = 0; o < R; ++o)
#pragma unroll
      for (int q = 0; q < Q; ++q) acc[o][q] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int c = 0; c < nch; ++c) {
      __syncthreads();  // the previous item's LDS reads (and the weight stores) are done
#pragma unroll
      for (int r = 0; r < kXLd; ++r)
        if ((live >> r) & 1) *(bf16x8*)(sIn + sbase + 8192 * r) = ld[r];
      if constexpr (STREAM) {
#pragma unroll
        for (int r = 0; r < kXWLd; ++r)
          if ((tid >> 8) + 2 * r < 9) *(bf16x8*)(sW + sbase + 8192 * r) = wl[r];
      }
      __syncthreads();
      {  // the next item's loads, in flight during this item's MFMAs
        int nt = tile, nc = c + 1;
        if (nc >= nch) {
          nt = tile + gridDim.x;
          nc = 0;
        }
        if (nt < ntiles) load_item(nt, nc * 32);
      }
      const char* wch = STREAM ? sW : sW + c * 9 * NCO * 64;
#pragma unroll
      for (int dx = 0; dx < 3; ++dx) {
        bf16x8 wf[3][Q];
#pragma unroll
        for (int dy = 0; dy < 3; ++dy)
#pragma unroll
          for (int q = 0; q < Q; ++q)
            wf[dy][q] = *(const bf16x8*)(wch + wbase + ((3 * dy + dx) * NCO + 16 * q) * 64);
#pragma unroll
        for (int r = 0; r < R + 2; ++r) {
          const bf16x8 pf = *(const bf16x8*)(sIn + pbase[dx] + r * kXPitch * 64);
#pragma unroll
          for (int o = 0; o < R; ++o) {
            const int dy = r - o;
            if (dy < 0 || dy > 2) continue;
#pragma unroll
            for (int q = 0; q < Q; ++q)
              acc[o][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[dy][q], pf, acc[o][q], 0, 0, 0);
          }
        }
      }
    }
    const int img = tile / (tilesx * tilesy);
    const int y0 = ((tile / tilesx) % tilesy) * kXTileH, x0 = (tile % tilesx) * kXTileW;
    const int x = x0 + 16 * wc + lr;
    float bv[Q][4];
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        bv[q][j] = MODE == 0 ? bias[min(co0 + q * 16 + 4 * lk + j, Cout - 1)] : 0.f;
#pragma unroll
    for (int o = 0; o < R; ++o) {
      const int y = y0 + 4 * wr + o;
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int cb = co0 + q * 16 + 4 * lk;
        if (x >= W || cb >= Cout) continue;
        const size_t off = (((size_t)img * H + y) * W + x) * Cout + cb;
        bf16x4 out;
        bf16x4 mk;
        if (MODE == 1 && mask) mk = *(const bf16x4*)(mask + off);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float v = acc[o][q][j];
          if (MODE == 0) {
            v = fmaxf(v + bv[q][j], 0.f);
          } else if (mask) {
            v = ((float)mk[j] > 0.f) ? v : 0.f;
          }
          out[j] = (__bf16)v;
        }
        *(bf16x4*)(Y + off) = out;
      }
    }
    if constexpr (MODE == 0) {
      if (pool) {  // fused 2 x 2 max-pool (H, W even; rows y0 + 4 wr + o, o even, pair up)
        const int H2 = H >> 1, W2 = W >> 1;
#pragma unroll
        for (int o = 0; o < R; o += 2) {
          const int y2 = (y0 + 4 * wr + o) >> 1;
#pragma unroll
          for (int q = 0; q < Q; ++q) {
            const int cb = co0 + q * 16 + 4 * lk;
            const bf16x4 m = pool_pair(acc[o][q], acc[o + 1][q], bv[q]);
            if (!(lr & 1) && x < W && cb < Cout)
              *(bf16x4*)(pool + (((size_t)img * H2 + y2) * W2 + (x >> 1)) * Cout + cb) = m;
          }
        }
      }
    }
  }
}

// ------------------------------------------------------------------------
// Weight and bias gradient of a 3x3 convolution: dW[co][t][ci] += sum_p
// dY[p][co] * X[p + off_t][ci], db[co] += sum_p dY[p][co], on BF16 MFMA with
// the pixels as the contraction axis.
//
// A wave owns a 32 x 32 (co, ci) block of ALL nine taps (144 accumulator
// registers) over a strip 32 pixels wide, and marches down the strip's rows:
// per input row it reads one new dY row (the two before stay in registers)
// and the input row once per tap column dx, and issues all 36 MFMAs of the
// nine taps on them, so dY and X are read once per (co, ci) tile instead of
// once per tap.  NHWC rows are staged in LDS as they lie in memory; the MFMA
// operands (8 pixels of one channel per lane) come out of LDS through the
// transposing read ds_read_b64_tr_b16, which takes a 4-pixel x 16-channel
// block per 16 lanes, so no transposed copy is written.  The order of the 32
// pixels along K is the same permutation for both operands.
// LDS pixels are 32 ch + 16 elements apart: the four pixels of a 16-lane read
// then lie in four different 32-byte bank groups.
//
// Workgroup: MB x NB blocks of 32 x 32 channels times S strips (one wave
// each); R rows are staged at a time, double-buffered, the next rows' global
// loads in flight during the MFMAs.  The rows of all images are one sequence
// with a zero row after each image (img * (H + 1) + y), cut into chunks, one
// per workgroup, so the launch fills the chip whatever n, H and W are.  The
// strips of a workgroup are summed through LDS; every workgroup stores its sum
// as one partial (in accumulator order, 256-byte runs) and dw_reduce_kernel
// adds the partials in a fixed order and writes the gradients: FP32 atomics on
// the shared gradient from every workgroup took longer than the MFMAs (64 -> 64
// at half resolution 116 us against 40).
// Bound at full resolution (32 channels) by memory, above it by LDS reads
// (16 transposing reads per 36 MFMAs) and the MFMAs.  16 images of 256 x 256,
// against a tap at a time with operands transposed by 2-byte LDS stores: 32 ->
// 32 at full resolution 699 -> 44 us (128 MB, 2.9 TB/s), 64 -> 64 at half 232
// -> 40 us, 384 -> 128 at quarter 494 -> 91 us (0.64 PFLOP/s), 256 -> 256 at an
// eighth 227 -> 62 us.
constexpr int kGrStrip = 32;

__device__ __forceinline__ bf16x8 lds_tr8(const __bf16* p0, const __bf16* p1) {
  typedef short v4s __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) v4s* lp;
  union {
    v4s h[2];
    bf16x8 v;
  } u;
  u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)p0);
  u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)p1);
  return u.v;
}

template <int MB, int NB, int S, int R>
struct GradConv {
  static constexpr int Threads = 64 * MB * NB * S;
  static constexpr int XP = 32 * NB + 16, YP = 32 * MB + 16;  // LDS pixel pitch (elements)
  static constexpr int XW = kGrStrip * S + 2, YW = kGrStrip * S;
  static constexpr int XRow = XW * XP, YRow = YW * YP;        // elements
  static constexpr int Stage = R * (XRow + YRow);
  static constexpr int XSlots = XW * NB * 4, YSlots = YW * MB * 4;  // 16-byte slots of a row
  static constexpr int XLd = (XSlots + Threads - 1) / Threads;
  static constexpr int YLd = (YSlots + Threads - 1) / Threads;
  static constexpr int Blocks = MB * NB;             // 32 x 32 blocks of a tile
  // strip sums go through LDS, one tap at a time, after the main loop
  static_assert(MB * NB * (S - 1) * 4096 <= 2 * Stage * 2, "strip sums fit the stages");
};

template <int MB, int NB, int S, int R>
__global__ __launch_bounds__(64 * MB * NB * S, 2) void conv3_dw_kernel(
    const __bf16* __restrict__ dY, int Cout, const __bf16* __restrict__ X1, int C1,
    const __bf16* __restrict__ X2, int C2, float* __restrict__ part, int n, int H, int W,
    int rows_per_wg, int strips_per_wg) {
  using G = GradConv<MB, NB, S, R>;
  __shared__ __attribute__((aligned(16))) __bf16 sm[2][G::Stage];
  const int Cin = C1 + C2;
  const int ncx = Cin / (32 * NB);
  const int co0 = (blockIdx.y / ncx) * 32 * MB, ci0 = (blockIdx.y % ncx) * 32 * NB;
  const int V = n * (H + 1);  // rows of all images, each followed by a zero row
  const int v0 = blockIdx.x * rows_per_wg, v1 = min(V, v0 + rows_per_wg);
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  const int s = wave / (MB * NB), wm = (wave / NB) % MB, wn = wave % NB;
  // the source of this workgroup's input channels (never straddles the two)
  const bool low = ci0 >= C1;
  const __bf16* __restrict__ X = low ? X2 + (ci0 - C1) : X1 + ci0;
  const int Cx = low ? C2 : C1, sh = low ? 1 : 0, Hx = H >> sh, Wx = W >> sh;

  // this thread's slots of a row: element offset in the source row, LDS
  // offset, and whether the pixel is in the image
  int xo[G::XLd], yo[G::YLd];
  unsigned xin = 0, yin = 0;
  auto slots = [&](int x0) {
    xin = yin = 0;
#pragma unroll
    for (int k = 0; k < G::XLd; ++k) {
      const int i = tid + G::Threads * k, px = i / (NB * 4), g = i % (NB * 4), x = x0 - 1 + px;
      xin |= (x >= 0 && x < W ? 1u : 0u) << k;
      xo[k] = (min(max(x, 0), W - 1) >> sh) * Cx + g * 8;
    }
#pragma unroll
    for (int k = 0; k < G::YLd; ++k) {
      const int i = tid + G::Threads * k, px = i / (MB * 4), g = i % (MB * 4), x = x0 + px;
      yin |= (x < W ? 1u : 0u) << k;
      yo[k] = min(x, W - 1) * Cout + co0 + g * 8;
    }
  };
  bf16x8 lx[R][G::XLd], ly[R][G::YLd];
  // input rows v .. v + R - 1 and the dY rows one below them
  auto load = [&](int v) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int vi = v + r, vo = vi + 1;
      const int im = max(vi, 0) / (H + 1), y = vi - im * (H + 1);
      const bool live = vi >= 0 && vi < V && y < H;  // uniform
      const __bf16* b = X + ((size_t)min(im, n - 1) * Hx + (min(max(y, 0), H - 1) >> sh)) * Wx * Cx;
#pragma unroll
      for (int k = 0; k < G::XLd; ++k) {
        const bf16x8 t = *(const bf16x8*)(b + xo[k]);
        lx[r][k] = live && ((xin >> k) & 1) ? t : zero8();
      }
      const int om = vo / (H + 1), q = vo - om * (H + 1);
      const bool olive = vo < v1 && q < H;  // vo >= v0 always
      const __bf16* d = dY + ((size_t)min(om, n - 1) * H + min(q, H - 1)) * W * Cout;
#pragma unroll
      for (int k = 0; k < G::YLd; ++k) {
        const bf16x8 t = *(const bf16x8*)(d + yo[k]);
        ly[r][k] = olive && ((yin >> k) & 1) ? t : zero8();
      }
    }
  };
  auto store = [&](__bf16* buf) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      __bf16* bx = buf + r * (G::XRow + G::YRow);
      __bf16* by = bx + G::XRow;
#pragma unroll
      for (int k = 0; k < G::XLd; ++k) {
        const int i = tid + G::Threads * k;
        if (i < G::XSlots) *(bf16x8*)(bx + (i / (NB * 4)) * G::XP + (i % (NB * 4)) * 8) = lx[r][k];
      }
#pragma unroll
      for (int k = 0; k < G::YLd; ++k) {
        const int i = tid + G::Threads * k;
        if (i < G::YSlots) *(bf16x8*)(by + (i / (MB * 4)) * G::YP + (i % (MB * 4)) * 8) = ly[r][k];
      }
    }
  };

  floatx4 acc[9][2][2], accb[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    accb[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int t = 0; t < 9; ++t) acc[t][i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  }
  bf16x8 a0[2], a1[2], a2[2], ones;  // dY rows vi - 1, vi, vi + 1
#pragma unroll
  for (int i = 0; i < 8; ++i) ones[i] = (__bf16)1.f;
  const bool bias = ci0 == 0 && wn == 0;
  // transposing read: lane l of a 16-lane group addresses pixel l / 4, channels
  // 4 (l % 4) .. + 3, and receives channel l of the four pixels; group lk reads
  // pixels 4 lk + (0..3) and, for the second half of K, 16 + 4 lk + (0..3)
  const int lpx = 4 * (lane / 16) + (lane % 16) / 4, lch = (lane % 4) * 4;
  const int xbase = (kGrStrip * s + lpx) * G::XP + wn * 32 + lch;
  const int ybase = (kGrStrip * s + lpx) * G::YP + wm * 32 + lch;

  const int strips = (W + kGrStrip * S - 1) / (kGrStrip * S);
  const int z1 = min(strips, ((int)blockIdx.z + 1) * strips_per_wg);
  for (int z = blockIdx.z * strips_per_wg; z < z1; ++z) {
    slots(z * kGrStrip * S);
#pragma unroll
    for (int i = 0; i < 2; ++i) a1[i] = a2[i] = zero8();
    load(v0 - 1);
    store(sm[0]);
    __syncthreads();
    int cur = 0;
    for (int v = v0 - 1; v <= v1; v += R, cur ^= 1) {
      const bool more = v + R <= v1;
      if (more) load(v + R);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const __bf16* bx = sm[cur] + r * (G::XRow + G::YRow) + xbase;
        const __bf16* by = sm[cur] + r * (G::XRow + G::YRow) + G::XRow + ybase;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          a0[i] = a1[i];
          a1[i] = a2[i];
          a2[i] = lds_tr8(by + i * 16, by + i * 16 + 16 * G::YP);
        }
        if (bias) {
#pragma unroll
          for (int i = 0; i < 2; ++i)
            accb[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2[i], ones, accb[i], 0, 0, 0);
        }
#pragma unroll
        for (int dx = 0; dx < 3; ++dx) {
          bf16x8 b[2];
#pragma unroll
          for (int j = 0; j < 2; ++j)
            b[j] = lds_tr8(bx + dx * G::XP + j * 16, bx + (dx + 16) * G::XP + j * 16);
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              // output row one below, at and above the input row: tap rows 0, 1, 2
              acc[dx][i][j] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2[i], b[j], acc[dx][i][j], 0, 0, 0);
              acc[3 + dx][i][j] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[i], b[j], acc[3 + dx][i][j], 0, 0, 0);
              acc[6 + dx][i][j] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[i], b[j], acc[6 + dx][i][j], 0, 0, 0);
            }
        }
      }
      if (more) store(sm[cur ^ 1]);
      __syncthreads();
    }
  }
  // acc[t][i][j][r]: co = co0 + 32 wm + 16 i + 4 lk + r, ci = ci0 + 32 wn + 16 j + lr;
  // partial: [tile][block][tap][16 registers][lane], then the biases [Cout]
  const int lr = lane % 16, lk = lane / 16;
  float* red = (float*)&sm[0][0];
  const int blk = wave % G::Blocks;
  const size_t pstride = (size_t)Cout * 9 * Cin + Cout;
  part += ((size_t)blockIdx.z * gridDim.x + blockIdx.x) * pstride;
  float* out = part + ((size_t)blockIdx.y * G::Blocks + blk) * 9 * 1024 + lane;
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    if (s > 0) {
      float* o = red + ((s - 1) * G::Blocks + blk) * 1024 + lane;
#pragma unroll
      for (int k = 0; k < 16; ++k) o[64 * k] = acc[t][k / 8][(k / 4) % 2][k % 4];
    }
    __syncthreads();
    if (s == 0) {
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        float v = acc[t][k / 8][(k / 4) % 2][k % 4];
#pragma unroll
        for (int q = 0; q < S - 1; ++q) v += red[(q * G::Blocks + blk) * 1024 + 64 * k + lane];
        out[(16 * t + k) * 64] = v;
      }
    }
    __syncthreads();
  }
  if (ci0 == 0) {
    if (bias && lr == 0) {
#pragma unroll
      for (int k = 0; k < 8; ++k)
        red[s * 32 * MB + 32 * wm + 16 * (k / 4) + 4 * lk + k % 4] = accb[k / 4][k % 4];
    }
    __syncthreads();
    if (tid < 32 * MB) {
      float v = 0.f;
#pragma unroll
      for (int q = 0; q < S; ++q) v += red[q * 32 * MB + tid];
      part[(size_t)Cout * 9 * Cin + co0 + tid] = v;
    }
  }
}

// Sum of np partials of conv3_dw_kernel<MB, NB, ...>, four consecutive values
// per thread: 16 threads read a partial's 256-byte run, 16 slices of partials
// per workgroup run side by side (the number of values alone would leave most
// CUs idle: 9 k for a 32 x 32 layer) and meet in LDS.
template <int MB, int NB>
__global__ __launch_bounds__(256) void dw_reduce_kernel(const float* __restrict__ part, int np,
                                                        float* __restrict__ dW,
                                                        float* __restrict__ db, int Cout,
                                                        int Cin) {
  __shared__ floatx4 red[16][16];
  const long nw = (long)Cout * 9 * Cin, count = nw + Cout;
  const int col = threadIdx.x % 16, slice = threadIdx.x / 16;
  const long i = ((long)blockIdx.x * 16 + col) * 4;
  floatx4 v{0.f, 0.f, 0.f, 0.f};
  if (i < count) {
#pragma unroll 4
    for (int p = slice; p < np; p += 16) v += *(const floatx4*)(part + p * (size_t)count + i);
  }
  red[slice][col] = v;
  __syncthreads();
  if (slice != 0 || i >= count) return;
#pragma unroll
  for (int q = 1; q < 16; ++q) v += red[q][col];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const long e = i + j;
    if (e >= nw) {
      db[e - nw] = v[j];
      continue;
    }
    const int lane = (int)(e % 64), k = (int)(e / 64 % 16), t = (int)(e / 1024 % 9);
    const int b = (int)(e / 9216), blk = b % (MB * NB), tile = b / (MB * NB);
    const int ncx = Cin / (32 * NB);
    const int co = ((tile / ncx) * MB + blk / NB) * 32 + 16 * (k / 8) + 4 * (lane / 16) + k % 4;
    const int ci = ((tile % ncx) * NB + blk % NB) * 32 + 16 * ((k / 4) % 2) + lane % 16;
    dW[((size_t)co * 9 + t) * Cin + ci] = v[j];
  }
}

// Orders LDS accesses between the lanes of one wave (its LDS traffic is
// processed in order; this keeps the compiler from moving it).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ------------------------------------------------------------------------
// Input layer: 2 channels (x = (cos, sin), float2) -> C0 channels, 3x3, relu.
// One thread per pixel computing all C0 outputs (the 9 neighbours are loaded
// once).
__global__ __launch_bounds__(256) void conv3_in_kernel(const float2* __restrict__ x,
                                                       const float* __restrict__ w,
                                                       const float* __restrict__ b,
                                                       __bf16* __restrict__ Y, int n, int H,
                                                       int W, int C0) {
  // the weights and biases are read at wave-uniform addresses straight from
  // global memory: the compiler turns them into scalar loads (SGPR operands of
  // the FMAs) instead of one LDS read per multiply-add
  // a wave's 64 pixels x 32 channels meet in LDS, so that each store writes 1 KB
  // of consecutive 16-byte pieces (one pixel per lane strides 2 C0 bytes); piece
  // g of pixel i sits at slot g ^ ((i >> 2) & 3), free of bank conflicts.  1 M
  // pixels, 32 channels: 36.4 -> 33.2 us (two pixels per lane, for half the
  // scalar weight loads per FMA, 34.1)
  __shared__ bf16x8 st[4][256];
  const int lane = threadIdx.x % 64;
  bf16x8* sw = st[threadIdx.x / 64];
  const long w0 = (long)blockIdx.x * blockDim.x + (threadIdx.x - lane);  // the wave's first pixel
  const long P = (long)n * H * W;
  if (w0 >= P) return;  // whole waves
  const long p = min(w0 + lane, P - 1);
  const int xx = (int)(p % W), yy = (int)((p / W) % H), img = (int)(p / ((long)W * H));
  // the nine taps are loaded from clamped (in-image) pixels without branches,
  // so all nine loads are in flight together, then zeroed outside the image
  float in[18];
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    const int y2 = yy + t / 3 - 1, x2 = xx + t % 3 - 1;
    const bool inside = y2 >= 0 && y2 < H && x2 >= 0 && x2 < W;
    const int yc = min(max(y2, 0), H - 1), xc = min(max(x2, 0), W - 1);
    const float2 v = x[((size_t)img * H + yc) * W + xc];
    in[2 * t] = inside ? v.x : 0.f;
    in[2 * t + 1] = inside ? v.y : 0.f;
  }
  for (int cb = 0; cb < C0; cb += 32) {
    for (int g = 0; g < 4; ++g) {
      bf16x8 o;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int co = cb + g * 8 + k;
        float s = b[co];
#pragma unroll
        for (int i = 0; i < 18; ++i) s = fmaf(w[co * 18 + i], in[i], s);
        o[k] = (__bf16)fmaxf(s, 0.f);
      }
      sw[lane * 4 + (g ^ ((lane >> 2) & 3))] = o;
    }
    wave_lds_sync();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int q = i * 64 + lane, px = q >> 2, g = q & 3;
      const bf16x8 v = sw[px * 4 + (g ^ ((px >> 2) & 3))];
      if (w0 + px < P) *(bf16x8*)(Y + (size_t)(w0 + px) * C0 + cb + g * 8) = v;
    }
    wave_lds_sync();
  }
}

// One halving step per lane bit (from bit O down to 1) of a sum over the
// wave's lanes of N values each: the lanes with the bit set keep the upper
// half (rounded up) of the values, the others the lower.  `at` collects the
// index of the lane's first remaining value, `cnt` how many it has (an odd
// count leaves the upper half one short).
template <int N, int O>
__device__ __forceinline__ void lane_fold(float* v, int lane, int& at, int& cnt) {
  constexpr int M = (N + 1) / 2;
  const bool up = lane & O;
#pragma unroll
  for (int i = 0; i < M; ++i) {
    const float hi = i + M < N ? v[i + M] : 0.f;
    const float keep = up ? hi : v[i], give = up ? v[i] : hi;
    v[i] = keep + __shfl_xor(give, O);
  }
  at += up ? M : 0;
  cnt = up ? max(cnt - M, 0) : min(cnt, M);
  if constexpr (O > 1) lane_fold<M, O / 2>(v, lane, at, cnt);
}

// weight/bias gradient of the input layer: dW[co][t][c] = sum_p dY[p][co]
// x[p+off_t][c].  FP32 on the vector ALU (x stays FP32).  A lane walks pixels
// of its row with 4 channels x (18 weights + bias) sums in registers: 76 FMAs
// on 9 + 1 loads, against two loads per FMA with one thread per weight (8
// channels a lane spill at two waves per SIMD).  The eight waves of a
// workgroup take the eight 4-channel groups of 32 channels, so together they
// read whole lines of dY.  A wave's sums meet through lane swaps at the
// end and go out as one partial per workgroup (partials_kernel adds them:
// atomics on the 608 shared sums serialised); 16 images of 256 x 256: 1690 ->
// 54 us.  Bound by the FMAs (16 us at 1 M pixels
// and 32 channels) and the 72 MB read.
__global__ __launch_bounds__(512, 4) void conv3_in_dw_kernel(const float2* __restrict__ x,
                                                             const __bf16* __restrict__ dY,
                                                             float* __restrict__ part, int n,
                                                             int H, int W, int C0) {
  const int lane = threadIdx.x % 64, co = blockIdx.y * 32 + (threadIdx.x / 64) * 4;
  const int rows = n * H;
  float acc[4][19];
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int i = 0; i < 19; ++i) acc[k][i] = 0.f;
  for (int r = blockIdx.x; r < rows; r += gridDim.x) {
    const int y = r % H;  // the row's image starts at row r - y
    const float2* xr[3];
    bool up[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int y2 = y + d - 1;
      up[d] = y2 >= 0 && y2 < H;
      xr[d] = x + (size_t)(r - y + min(max(y2, 0), H - 1)) * W;
    }
    for (int xx = lane; xx < W; xx += 64) {
      float in[18];
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        const int x2 = xx + t % 3 - 1;
        const float2 v = xr[t / 3][min(max(x2, 0), W - 1)];
        const bool inside = up[t / 3] && x2 >= 0 && x2 < W;
        in[2 * t] = inside ? v.x : 0.f;
        in[2 * t + 1] = inside ? v.y : 0.f;
      }
      const bf16x4 g4 = *(const bf16x4*)(dY + ((size_t)r * W + xx) * C0 + co);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float g = (float)g4[k];
#pragma unroll
        for (int i = 0; i < 18; ++i) acc[k][i] = fmaf(g, in[i], acc[k][i]);
        acc[k][18] += g;
      }
    }
  }
  // sum over the wave's lanes by halving: at each step a lane hands half of its
  // values to its partner and adds the partner's share of the other half (77
  // exchanges for 76 sums instead of six each)
  float v[76];
#pragma unroll
  for (int i = 0; i < 76; ++i) v[i] = acc[i / 19][i % 19];
  int at = 0, cnt = 76;
  lane_fold<76, 32>(v, lane, at, cnt);
  part += (size_t)blockIdx.x * C0 * 19;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int i = at + q, k = i / 19, w = i % 19;
    if (q < cnt) part[w == 18 ? C0 * 18 + co + k : (co + k) * 18 + w] = v[q];
  }
}

// out0[n0], out1[n1], out2[n2] = the sums over np partials of n0 + n1 + n2
// consecutive values (pitch floats apart), in a fixed order: 16 values side by
// side, 16 slices of partials per workgroup.
__global__ __launch_bounds__(256) void partials_kernel(const float* __restrict__ part, int np,
                                                       int pitch, float* __restrict__ out0, int n0,
                                                       float* __restrict__ out1, int n1,
                                                       float* __restrict__ out2, int n2) {
  __shared__ float red[16][17];
  const int col = threadIdx.x % 16, slice = threadIdx.x / 16, i = blockIdx.x * 16 + col;
  float v = 0.f;
  if (i < n0 + n1 + n2) {
#pragma unroll 8
    for (int p = slice; p < np; p += 16) v += part[(size_t)p * pitch + i];
  }
  red[slice][col] = v;
  __syncthreads();
  if (slice != 0 || i >= n0 + n1 + n2) return;
#pragma unroll
  for (int q = 1; q < 16; ++q) v += red[q][col];
  if (i < n0) out0[i] = v;
  else if (i < n0 + n1) out1[i - n0] = v;
  else out2[i - n0 - n1] = v;
}

// ------------------------------------------------------------------------
// Output layer: out = x + W d + b (1x1, C0 -> 2), FP32.
__global__ __launch_bounds__(256) void conv1_out_kernel(const __bf16* __restrict__ d,
                                                        const float2* __restrict__ x,
                                                        const float* __restrict__ w,
                                                        const float* __restrict__ b,
                                                        float2* __restrict__ out, long P, int C0) {
  const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P) return;
  float s0 = b[0], s1 = b[1];
  for (int c = 0; c < C0; c += 8) {
    const bf16x8 v = *(const bf16x8*)(d + (size_t)p * C0 + c);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float f = (float)v[k];
      s0 = fmaf(w[c + k], f, s0);
      s1 = fmaf(w[C0 + c + k], f, s1);
    }
  }
  const float2 xi = x[p];
  out[p] = make_float2(xi.x + s0, xi.y + s1);
}

// Loss L = mean |out - u|^2 and its backward through the output layer:
// g = 2 (out - u) / P; dd = (W^T g) * (d > 0); dW += g d^T; db += g.
// Four threads per pixel, 8 channels each (32 channels per blockIdx.y), so d
// and dd move in 16-byte pieces of whole lines; every thread keeps its 16
// weight sums (and the loss and bias sums) in registers over a grid-stride
// walk and the workgroup reduces once at the end, instead of a workgroup-wide
// reduction per channel for every 256 pixels; partials_kernel adds the
// workgroups' partials (atomics on the 67 shared sums serialised: more
// workgroups made the kernel slower).  16 images of 256 x 256: 1650 -> 32 us.
// Bound by memory: 144 MB at 1 M pixels and 32 channels, 4.5 TB/s.
__global__ __launch_bounds__(256) void conv1_out_bwd_kernel(
    const __bf16* __restrict__ d, const float2* __restrict__ out, const float2* __restrict__ u,
    const float* __restrict__ w, __bf16* __restrict__ dd, float* __restrict__ part, long P,
    int C0) {
  __shared__ float red[4][4][19];  // [wave][channel group][sum]
  const int g = threadIdx.x % 4, lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int c0 = blockIdx.y * 32 + 8 * g;
  const float invP = 1.f / (float)P;
  float w0[8], w1[8], s[19];  // s: dW[0][8], dW[1][8], loss, db[0], db[1]
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    w0[k] = w[c0 + k];
    w1[k] = w[C0 + c0 + k];
  }
#pragma unroll
  for (int k = 0; k < 19; ++k) s[k] = 0.f;
  for (long p = (long)blockIdx.x * 64 + threadIdx.x / 4; p < P; p += (long)gridDim.x * 64) {
    const float2 o = out[p], t = u[p];
    const bf16x8 v = *(const bf16x8*)(d + (size_t)p * C0 + c0);
    const float r0 = o.x - t.x, r1 = o.y - t.y;
    const float g0 = 2.f * r0 * invP, g1 = 2.f * r1 * invP;
    s[16] += (r0 * r0 + r1 * r1) * invP;
    s[17] += g0;
    s[18] += g1;
    bf16x8 q;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float f = (float)v[k];
      q[k] = (__bf16)(f > 0.f ? w0[k] * g0 + w1[k] * g1 : 0.f);
      s[k] = fmaf(g0, f, s[k]);
      s[8 + k] = fmaf(g1, f, s[8 + k]);
    }
    *(bf16x8*)(dd + (size_t)p * C0 + c0) = q;
  }
#pragma unroll
  for (int k = 0; k < 19; ++k) {
    float v = s[k];
#pragma unroll
    for (int o = 32; o >= 4; o >>= 1) v += __shfl_xor(v, o);
    if (lane < 4) red[wave][lane][k] = v;
  }
  __syncthreads();
  if (threadIdx.x < 76) {
    const int h = threadIdx.x / 19, k = threadIdx.x % 19, c = blockIdx.y * 32 + 8 * h;
    const float v = red[0][h][k] + red[1][h][k] + red[2][h][k] + red[3][h][k];
    // partial: dW [2][C0], db [2], loss
    part += (size_t)blockIdx.x * (2 * C0 + 3);
    if (k < 8) part[c + k] = v;
    else if (k < 16) part[C0 + c + k - 8] = v;
    else if (h == 0 && blockIdx.y == 0) part[2 * C0 + (k == 16 ? 2 : k - 17)] = v;
  }
}

// ------------------------------------------------------------------------
__global__ __launch_bounds__(256) void maxpool2_kernel(const __bf16* __restrict__ x,
                                                       __bf16* __restrict__ y, int n, int H,
                                                       int W, int C) {
  const int H2 = H / 2, W2 = W / 2, G = C / 8;
  const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= (long)n * H2 * W2 * G) return;
  const int g = (int)(gid % G);
  const long q = gid / G;
  const int x2 = (int)(q % W2), y2 = (int)((q / W2) % H2), img = (int)(q / ((long)W2 * H2));
  const __bf16* b = x + (((size_t)img * H + 2 * y2) * W + 2 * x2) * C + g * 8;
  const bf16x8 v0 = *(const bf16x8*)b, v1 = *(const bf16x8*)(b + C);
  const bf16x8 v2 = *(const bf16x8*)(b + (size_t)W * C), v3 = *(const bf16x8*)(b + (size_t)W * C + C);
  bf16x8 o;
#pragma unroll
  for (int k = 0; k < 8; ++k)
    o[k] = (__bf16)fmaxf(fmaxf((float)v0[k], (float)v1[k]), fmaxf((float)v2[k], (float)v3[k]));
  *(bf16x8*)(y + (size_t)q * C + g * 8) = o;
}

// Gradient into an encoder output e (C channels, H x W) from its two
// consumers, then through its relu:  g_e = (pool adjoint of gp (H/2 x W/2)
// routed to the first maximum of each window, row-major) + gskip (channels
// [0, C) of the decoder's concatenated input gradient, pitch Cs), times
// (e > 0).  One thread per window and 8 channels (16-byte accesses; one
// channel per thread moved 2 bytes at a time: 82 -> 52 us on 16 images of 256 x
// 256, 32 channels).  Bound by memory.
__global__ __launch_bounds__(256) void pool_bwd_kernel(const __bf16* __restrict__ e,
                                                       const __bf16* __restrict__ gp,
                                                       const __bf16* __restrict__ gskip, int Cs,
                                                       __bf16* __restrict__ ge, int n, int H,
                                                       int W, int C) {
  const int H2 = H / 2, W2 = W / 2, G = C / 8;
  const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= (long)n * H2 * W2 * G) return;
  const int c = (int)(gid % G) * 8;
  const long q = gid / G;
  const int x2 = (int)(q % W2), y2 = (int)((q / W2) % H2), img = (int)(q / ((long)W2 * H2));
  const bf16x8 g = *(const bf16x8*)(gp + q * C + c);
  bf16x8 ev[4], gs[4];
  size_t pix[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    pix[k] = ((size_t)img * H + 2 * y2 + k / 2) * W + 2 * x2 + k % 2;
    ev[k] = *(const bf16x8*)(e + pix[k] * C + c);
    gs[k] = *(const bf16x8*)(gskip + pix[k] * Cs + c);
  }
  bf16x8 o[4];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    float best = (float)ev[0][j];
    int arg = 0;
#pragma unroll
    for (int k = 1; k < 4; ++k) {
      const float v = (float)ev[k][j];
      if (v > best) {
        best = v;
        arg = k;
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float v = (k == arg ? (float)g[j] : 0.f) + (float)gs[k][j];
      o[k][j] = (__bf16)((float)ev[k][j] > 0.f ? v : 0.f);
    }
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) *(bf16x8*)(ge + pix[k] * C + c) = o[k];
}

// Adjoint of the nearest x2 upsampling of a decoder input (channels [C1,
// C1+C) of the concatenated gradient gcat, full resolution, pitch C1 + C),
// times (a > 0) for the low-resolution activation a (C channels).  One thread
// per low-resolution pixel and 8 channels; bound by memory (67 -> 43 us on 16
// images of 256 x 256, 64 channels).
__global__ __launch_bounds__(256) void up_bwd_kernel(const __bf16* __restrict__ gcat, int C1,
                                                     const __bf16* __restrict__ a,
                                                     __bf16* __restrict__ ga, int n, int H2,
                                                     int W2, int C) {
  const int G = C / 8;
  const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= (long)n * H2 * W2 * G) return;
  const int c = (int)(gid % G) * 8;
  const long q = gid / G;
  const int x2 = (int)(q % W2), y2 = (int)((q / W2) % H2), img = (int)(q / ((long)W2 * H2));
  const int H = 2 * H2, W = 2 * W2, Cc = C1 + C;
  bf16x8 v[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const size_t pix = ((size_t)img * H + 2 * y2 + k / 2) * W + 2 * x2 + k % 2;
    v[k] = *(const bf16x8*)(gcat + pix * Cc + C1 + c);
  }
  const bf16x8 av = *(const bf16x8*)(a + q * C + c);
  bf16x8 o;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) s += (float)v[k][j];
    o[j] = (__bf16)((float)av[j] > 0.f ? s : 0.f);
  }
  *(bf16x8*)(ga + q * C + c) = o;
}

// Adam on FP32 master weights; refreshes the BF16 copies: Wf [Cout][9][Cin]
// and, for 3x3 layers, the flipped transpose Wt [Cin][9][Cout].
__global__ __launch_bounds__(256) void adam_kernel(float* __restrict__ w,
                                                   const float* __restrict__ g,
                                                   float* __restrict__ m, float* __restrict__ v,
                                                   long count, float lr, float b1, float b2,
                                                   float eps, float c1, float c2) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  w[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
}

__global__ __launch_bounds__(256) void weights_to_bf16_kernel(const float* __restrict__ w,
                                                              __bf16* __restrict__ wf,
                                                              __bf16* __restrict__ wt, int Cout,
                                                              int Cin) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)Cout * 9 * Cin) return;
  const int ci = (int)(i % Cin), t = (int)((i / Cin) % 9), co = (int)(i / (9L * Cin));
  const __bf16 h = (__bf16)w[i];
  wf[i] = h;
  if (wt) wt[((size_t)ci * 9 + (8 - t)) * Cout + co] = h;
}

// ======================================================== host launchers
static unsigned blocks(long work, int per = 256) { return (unsigned)((work + per - 1) / per); }

// CUs of the current device (0 on error); callable from several threads.
int unet_device_cus() {
  constexpr int kDevices = 64;
  static std::atomic<int> cus[kDevices] = {};
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kDevices) return 0;
  int v = cus[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      return 0;
    cus[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}

hipError_t unet_conv3(const __bf16* X1, int C1, const __bf16* X2, int C2, const __bf16* Wt,
                      const float* bias, const __bf16* mask, __bf16* Y, int n, int H, int W,
                      int Cout, int mode, hipStream_t s, __bf16* pool) {
  if ((C1 % 32) || (C2 % 32) || (Cout % 16) || (H % kTileH) || (C2 && ((H | W) & 1)) ||
      (pool && (mode != 0 || ((H | W) & 1))))
    return hipErrorInvalidValue;
  const int nco = Cout >= 64 ? 64 : 32;
  const int cob = (Cout + nco - 1) / nco;
  if (nco == 32 && H % kRTileH == 0) {
    // persistent 8-row kernel: two workgroups per CU (64 KB LDS, <= 256 registers)
    const int cus = unet_device_cus();
    if (cus < 1) return hipErrorInvalidValue;
    const int rtiles = n * (H / kRTileH) * ((W + RowsConv<32>::TW - 1) / RowsConv<32>::TW);
    dim3 grid(std::min(rtiles, std::max(1, 2 * cus / cob)), cob);
    if (mode == 0)
      hipLaunchKernelGGL((conv3_rows_kernel<32, 0>), grid, dim3(256), 0, s, X1, C1, X2, C2, Wt,
                         bias, mask, Y, n, H, W, Cout, pool);
    else
      hipLaunchKernelGGL((conv3_rows_kernel<32, 1>), grid, dim3(256), 0, s, X1, C1, X2, C2, Wt,
                         bias, mask, Y, n, H, W, Cout, nullptr);
    return hipGetLastError();
  }
  if (nco == 64 && H % kXTileH == 0) {
    // one 8-wave workgroup per CU: weights resident up to 64 input channels;
    // above that, for the forward pass, streamed per chunk where the tiles fill
    // every CU
    const int cus = unet_device_cus();
    if (cus < 1) return hipErrorInvalidValue;
    const int xt = n * (H / kXTileH) * ((W + kXTileW - 1) / kXTileW);
    const bool resident = C1 + C2 <= kXMaxCin;
    if (resident || (mode == 0 && xt * cob >= cus)) {
      dim3 gridx(std::min(xt, std::max(1, cus / cob)), cob);
#define GLSU_CONV3_RES64(MD, ST)                                                                 \
  hipLaunchKernelGGL((conv3_res64_kernel<MD, ST>), gridx, dim3(512), 0, s, X1, C1, X2, C2, Wt,   \
                     bias, mask, Y, n, H, W, Cout, pool)
      if (resident) {
        if (mode == 0) GLSU_CONV3_RES64(0, false);
        else GLSU_CONV3_RES64(1, false);
      } else {
        GLSU_CONV3_RES64(0, true);
      }
#undef GLSU_CONV3_RES64
      return hipGetLastError();
    }
  }

  const int tiles = n * (H / kTileH) * ((W + kTileW - 1) / kTileW);
  dim3 grid(tiles, cob);
  if (nco == 64) {
    if (mode == 0)
      hipLaunchKernelGGL((conv3_mfma_kernel<64, 0>), grid, dim3(256), 0, s, X1, C1, X2, C2, Wt,
                         bias, mask, Y, n, H, W, Cout);
    else
      hipLaunchKernelGGL((conv3_mfma_kernel<64, 1>), grid, dim3(256), 0, s, X1, C1, X2, C2, Wt,
                         bias, mask, Y, n, H, W, Cout);
  } else {
    if (mode == 0)
      hipLaunchKernelGGL((conv3_mfma_kernel<32, 0>), grid, dim3(256), 0, s, X1, C1, X2, C2, Wt,
                         bias, mask, Y, n, H, W, Cout);
    else
      hipLaunchKernelGGL((conv3_mfma_kernel<32, 1>), grid, dim3(256), 0, s, X1, C1, X2, C2, Wt,
                         bias, mask, Y, n, H, W, Cout);
  }
  // this kernel has no pooled epilogue
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || !pool) return e;
  return unet_maxpool2(Y, pool, n, H, W, Cout, s);
}

// Partition of one weight gradient: workgroups per (co, ci) tile along the
// rows and along the strips; their product is the number of partials.
struct DwSplit {
  int rows, chunks, strips, groups;  // rows per chunk, chunks, strips per group, groups
};
template <int MB, int NB, int S, int R>
static DwSplit dw_split(int Cout, int Cin, int n, int H, int W, int wgs) {
  const int tiles = (Cout / (32 * MB)) * (Cin / (32 * NB));
  const int ns = (W + kGrStrip * S - 1) / (kGrStrip * S);
  // as many partials as fill the chip once, but at least six rows each (every
  // chunk reads two input rows more than it owns)
  const int want = std::max(1, wgs / tiles), V = n * (H + 1);
  DwSplit d;
  const int g = std::min(ns, want);
  d.strips = (ns + g - 1) / g;
  d.groups = (ns + d.strips - 1) / d.strips;
  const int c = std::max(1, std::min(want / d.groups, V / 6));
  d.rows = (V + c - 1) / c;
  d.chunks = (V + d.rows - 1) / d.rows;
  return d;
}
template <int MB, int NB, int S, int R>
static hipError_t launch_dw(const __bf16* dY, int Cout, const __bf16* X1, int C1, const __bf16* X2,
                            int C2, float* dW, float* db, float* ws, int n, int H, int W, int wgs,
                            hipStream_t s) {
  const int Cin = C1 + C2, tiles = (Cout / (32 * MB)) * (Cin / (32 * NB));
  const DwSplit d = dw_split<MB, NB, S, R>(Cout, Cin, n, H, W, wgs);
  hipLaunchKernelGGL((conv3_dw_kernel<MB, NB, S, R>), dim3(d.chunks, tiles, d.groups),
                     dim3(GradConv<MB, NB, S, R>::Threads), 0, s, dY, Cout, X1, C1, X2, C2, ws, n,
                     H, W, d.rows, d.strips);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const long count = (long)Cout * 9 * Cin + Cout;
  hipLaunchKernelGGL((dw_reduce_kernel<MB, NB>), dim3(blocks(count, 64)), dim3(256), 0, s, ws,
                     d.chunks * d.groups, dW, db, Cout, Cin);
  return hipGetLastError();
}

// The widest channel tile that divides the layer: 64 x 64 reads each operand
// for two blocks; narrower layers share the workgroup's waves over strips.
static int dw_tile(int Cout, int C1, int C2) {
  if (Cout % 64) return 0;
  return C1 % 64 || C2 % 64 ? 1 : 2;
}

size_t unet_conv3_dw_floats(int Cout, int C1, int C2, int n, int H, int W, int cus) {
  const int Cin = C1 + C2;
  DwSplit d;
  switch (dw_tile(Cout, C1, C2)) {
    case 2: d = dw_split<2, 2, 2, 2>(Cout, Cin, n, H, W, cus); break;
    case 1: d = dw_split<2, 1, 4, 1>(Cout, Cin, n, H, W, cus); break;
    default: d = dw_split<1, 1, 4, 1>(Cout, Cin, n, H, W, 2 * cus); break;
  }
  return (size_t)d.chunks * d.groups * ((size_t)Cout * 9 * Cin + Cout);
}

hipError_t unet_conv3_dw(const __bf16* dY, int Cout, const __bf16* X1, int C1, const __bf16* X2,
                         int C2, float* dW, float* db, float* ws, int n, int H, int W, int cus,
                         hipStream_t s) {
  if ((C1 % 32) || (C2 % 32) || (Cout % 32) || (C2 && ((H | W) & 1)) || cus < 1)
    return hipErrorInvalidValue;
  switch (dw_tile(Cout, C1, C2)) {
    case 2:
      return launch_dw<2, 2, 2, 2>(dY, Cout, X1, C1, X2, C2, dW, db, ws, n, H, W, cus, s);
    case 1:
      return launch_dw<2, 1, 4, 1>(dY, Cout, X1, C1, X2, C2, dW, db, ws, n, H, W, cus, s);
    default:
      return launch_dw<1, 1, 4, 1>(dY, Cout, X1, C1, X2, C2, dW, db, ws, n, H, W, 2 * cus, s);
  }
}

hipError_t unet_conv3_in(const float2* x, const float* w, const float* b, __bf16* Y, int n,
                         int H, int W, int C0, hipStream_t s) {
  const long work = (long)n * H * W;
  hipLaunchKernelGGL(conv3_in_kernel, dim3(blocks(work)), dim3(256), 0, s, x, w, b, Y, n, H, W,
                     C0);
  return hipGetLastError();
}

// workgroups of conv3_in_dw_kernel (two per CU, rows dealt round robin)
static int in_dw_wgs(long rows, int C0, int cus) {
  return (int)std::max(1L, std::min<long>(rows, 2L * cus / (C0 / 32)));
}
size_t unet_conv3_in_dw_floats(int n, int H, int C0, int cus) {
  return (size_t)in_dw_wgs((long)n * H, C0, cus) * C0 * 19;
}
hipError_t unet_conv3_in_dw(const float2* x, const __bf16* dY, float* dW, float* db, float* ws,
                            int n, int H, int W, int C0, int cus, hipStream_t s) {
  if (C0 % 32 || cus < 1) return hipErrorInvalidValue;
  const int wgs = in_dw_wgs((long)n * H, C0, cus);
  hipLaunchKernelGGL(conv3_in_dw_kernel, dim3(wgs, C0 / 32), dim3(512), 0, s, x, dY, ws, n, H, W,
                     C0);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(partials_kernel, dim3(blocks(C0 * 19, 16)), dim3(256), 0, s, ws, wgs, C0 * 19,
                     dW, C0 * 18, db, C0, nullptr, 0);
  return hipGetLastError();
}

hipError_t unet_conv1_out(const __bf16* d, const float2* x, const float* w, const float* b,
                          float2* out, long P, int C0, hipStream_t s) {
  hipLaunchKernelGGL(conv1_out_kernel, dim3(blocks(P)), dim3(256), 0, s, d, x, w, b, out, P, C0);
  return hipGetLastError();
}

// workgroups of conv1_out_bwd_kernel (eight per CU walk the pixels)
static int out_bwd_wgs(long P, int C0, int cus) {
  return (int)std::max(1L, std::min<long>((P + 63) / 64, 8L * cus / (C0 / 32)));
}
size_t unet_conv1_out_bwd_floats(long P, int C0, int cus) {
  return (size_t)out_bwd_wgs(P, C0, cus) * (2 * C0 + 3);
}
hipError_t unet_conv1_out_bwd(const __bf16* d, const float2* out, const float2* u,
                              const float* w, __bf16* dd, float* dW, float* db, float* loss,
                              float* ws, long P, int C0, int cus, hipStream_t s) {
  if (C0 % 32 || cus < 1) return hipErrorInvalidValue;
  const int wgs = out_bwd_wgs(P, C0, cus);
  hipLaunchKernelGGL(conv1_out_bwd_kernel, dim3(wgs, C0 / 32), dim3(256), 0, s, d, out, u, w, dd,
                     ws, P, C0);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(partials_kernel, dim3(blocks(2 * C0 + 3, 16)), dim3(256), 0, s, ws, wgs,
                     2 * C0 + 3, dW, 2 * C0, db, 2, loss, 1);
  return hipGetLastError();
}

hipError_t unet_maxpool2(const __bf16* x, __bf16* y, int n, int H, int W, int C, hipStream_t s) {
  const long work = (long)n * (H / 2) * (W / 2) * (C / 8);
  hipLaunchKernelGGL(maxpool2_kernel, dim3(blocks(work)), dim3(256), 0, s, x, y, n, H, W, C);
  return hipGetLastError();
}

hipError_t unet_pool_bwd(const __bf16* e, const __bf16* gp, const __bf16* gskip, int Cs,
                         __bf16* ge, int n, int H, int W, int C, hipStream_t s) {
  const long work = (long)n * (H / 2) * (W / 2) * (C / 8);
  hipLaunchKernelGGL(pool_bwd_kernel, dim3(blocks(work)), dim3(256), 0, s, e, gp, gskip, Cs, ge,
                     n, H, W, C);
  return hipGetLastError();
}

hipError_t unet_up_bwd(const __bf16* gcat, int C1, const __bf16* a, __bf16* ga, int n, int H2,
                       int W2, int C, hipStream_t s) {
  const long work = (long)n * H2 * W2 * (C / 8);
  hipLaunchKernelGGL(up_bwd_kernel, dim3(blocks(work)), dim3(256), 0, s, gcat, C1, a, ga, n, H2,
                     W2, C);
  return hipGetLastError();
}

hipError_t unet_adam(float* w, const float* g, float* m, float* v, long count, float lr,
                     float b1, float b2, float eps, int step, hipStream_t s) {
  const float c1 = 1.f / (1.f - powf(b1, (float)step));
  const float c2 = 1.f / (1.f - powf(b2, (float)step));
  hipLaunchKernelGGL(adam_kernel, dim3(blocks(count)), dim3(256), 0, s, w, g, m, v, count, lr,
                     b1, b2, eps, c1, c2);
  return hipGetLastError();
}

hipError_t unet_weights_bf16(const float* w, __bf16* wf, __bf16* wt, int Cout, int Cin,
                             hipStream_t s) {
  hipLaunchKernelGGL(weights_to_bf16_kernel, dim3(blocks((long)Cout * 9 * Cin)), dim3(256), 0, s,
                     w, wf, wt, Cout, Cin);
  return hipGetLastError();
}

}  // namespace glsu
