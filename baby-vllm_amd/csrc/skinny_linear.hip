// Linear layers of a few tokens: out[m, c] = Σ_k x[m, k]·w[c, k] (+ bias[c]), and
// the gated form out[m, c] = silu(Σ x·w[c]) · Σ x·w[n + c] of an MLP's fused
// gate/up projection, for the decode steps of a model (reference: nn.Linear
// calls of babyvllm/models/qwen2.py:17-137).
//
// HBM-bound on the weights: at 16 tokens each weight is used 16 times, far
// below what MFMA could do, so the kernel is built to keep weight reads in
// flight on every CU and to feed x cheaply.
//
// Work-group = (row group, k split), RW·KW waves: wave (rw, kw) owns a tile of
// at most 16 weight rows and every KW-th slab of the work-group's k range, and
// streams its weights straight into MFMA operand registers (lane n + 16g holds
// 16 bytes of row n; four 64-byte pieces make a 256-byte stage of 128 k), D
// stages ahead. x passes through LDS: the RW waves of a slab load its
// [tokens, 128 k] stage once, whole 256-byte rows, 16-byte chunks XOR-swizzled by
// row so that writes and operand reads are conflict-free. (x read straight into
// operand registers costs as many L1 lookups per token tile as the weights
// do: 3584 x 18944, 16 tokens: 36.7 against 29 us.) Buffer loads with a
// zero-sized descriptor past a slab's end return zeros with no traffic, so the
// steady state has no branch around loads and the compiler's counted waits keep
// D stages in flight (D = 2: more put too many requests on HBM, 4 was slower at
// every shape). The KW partial sums meet in LDS in slab order; k splits over
// work-groups (few rows, long k) write fp32 partials that a second launch adds
// in split order. The same (w shape, 16-token tile count) always sums in the same
// order.
//
// Rows are cut evenly over a multiple of 256 work-groups instead of in
// tiles of 16·RW: with 592 or 296 work-groups the CUs holding one more than
// the others set the time (gate/up 37888 x 3584, 16 tokens: 56 -> 49.6 us).
//
// Measured against hipBLASLt (+ the SiLU·mul launch for gated), us, weights from
// HBM, graph of back-to-back calls:
//   gate/up 2·18944 x 3584: 1 token 56 + 3 -> 47, 16: 54 + 3 -> 50, 64: 60 + 3 -> 63
//   down 3584 x 18944:      16 tokens 48 -> 29, 32: 110 -> 32, 64: 91 -> 36, 128: 99 -> 47,
//                           256 (two blocks of 128 side by side, weights shared in cache): 126 -> 83
//   head 152064 x 3584:     1 token 228 -> 177, 16: 231 -> 188, 32: 250 -> 197
//   qkv 4608 x 3584:        16 tokens 12.3 -> 10.4;  out 3584 x 3584: 11.9 -> 9.6
#include "bvllm_device.h"
#include "bvllm_abi_internal.h"

#include <algorithm>
#include <type_traits>

namespace bvllm {

namespace {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

constexpr int kStageK = 128;  // k per stage: 256 bytes of a row
// Offset of a lane with nothing to load: past every descriptor's end (sizes stay
// below it, checked on the host), also after a stage offset is added.
constexpr uint32_t kNoLoad = 0x80000000u;

__device__ __forceinline__ float silu(float g) {
  return g * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(g * -kLog2e));
}

// First row of row group i of G: even split of n rows in units of `unit`.
__device__ __forceinline__ int group_row(int n, int unit, int i, int G) {
  return (int)((int64_t)(n / unit) * i / G) * unit;
}

__device__ __forceinline__ void store4(const LinearArgs& a, int m, int col, int col_end, f32x4_t y) {
  uint16_t* dst = reinterpret_cast<uint16_t*>(a.out) + (int64_t)m * a.out_stride + col;
  const uint32_t lo = pack_bf16x2_hw(y[0], y[1]), hi = pack_bf16x2_hw(y[2], y[3]);
  if (a.unit == 4) {  // uniform
    st8(dst, make_uint2(lo, hi));
  } else {
    *reinterpret_cast<uint32_t*>(dst) = lo;
    if (col + 2 < col_end) *reinterpret_cast<uint32_t*>(dst + 2) = hi;
  }
}

__device__ __forceinline__ f32x4_t add_bias(const LinearArgs& a, int col, int col_end, f32x4_t y) {
  if (a.bias != nullptr) {
    const uint16_t* b = reinterpret_cast<const uint16_t*>(a.bias) + col;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (col + i < col_end) y[i] += bf16_to_f32(b[i]);
  }
  return y;
}

// MT: 16-token tiles. GLU: waves rw < RW/2 take gate rows, the others the up
// rows of the same output columns.
template <int MT, int RW, int KW, int D, bool GLU>
__global__ __launch_bounds__(RW * KW * 64) void skinny_linear_kernel(LinearArgs a) {
  constexpr int NW = RW * KW;
  constexpr int XB = MT * 16 * 256;           // bytes of one slab's x stage
  constexpr int XL = (MT * 4 + RW - 1) / RW;  // x loads per lane and stage
  constexpr bool XALL = XL * RW == MT * 4;    // every lane has a row for every x load
  constexpr int CW = GLU ? RW / 2 : RW;       // 16-column tiles of the work-group
  constexpr int XLDS = 2 * KW * XB, RLDS = NW * MT * 1024;
  static_assert(!GLU || RW % 2 == 0, "gate and up waves come in pairs");
  __shared__ __attribute__((aligned(16))) unsigned char lds[XLDS > RLDS ? XLDS : RLDS];

  const int lane = lane_id(), n = lane & 15, g = lane >> 4, w = wave_id();
  const int rw = w % RW, kw = w / RW;
  const int ks = (int)blockIdx.x % a.k_splits, rg = (int)blockIdx.x / a.k_splits;
  const int m0 = (int)blockIdx.y * MT * 16, m_here = min(a.m - m0, MT * 16);  // the token block
  const int row0 = group_row(a.n, a.unit, rg, a.row_groups);
  const int row1 = group_row(a.n, a.unit, rg + 1, a.row_groups);

  // The wave's slab of stages, and the longest slab of the work-group (barriers).
  const int S = a.k / kStageK, parts = a.k_splits * KW;
  auto slab = [&](int p) { return (int)((int64_t)S * p / parts); };
  const int j0 = slab(ks * KW + kw), j1 = slab(ks * KW + kw + 1);
  int steps = 0;
#pragma unroll
  for (int q = 0; q < KW; ++q) steps = max(steps, slab(ks * KW + q + 1) - slab(ks * KW + q));

  const uint32_t w_bytes = (GLU ? 2u : 1u) * (uint32_t)a.n * (uint32_t)a.k * 2u;
  const uint32_t x_bytes = (uint32_t)m_here * (uint32_t)a.x_stride * 2u;
  const uint16_t* x = reinterpret_cast<const uint16_t*>(a.x) + (int64_t)m0 * a.x_stride;
  const int col = row0 + 16 * (rw % CW) + n;
  const uint32_t w_row = (uint32_t)(col + (GLU && rw >= CW ? a.n : 0));
  const uint32_t w_off = col < row1 ? w_row * (uint32_t)a.k * 2u + 16u * g : kNoLoad;
  uint32_t x_off[XL], x_dst[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int e = (i * RW + rw) * 64 + lane;  // row e / 16, chunk e mod 16; rows past m read as zeros
    const int r = e >> 4, c = e & 15;
    x_off[i] = r < m_here ? (uint32_t)r * (uint32_t)a.x_stride * 2u + 16u * c : kNoLoad;
    x_dst[i] = (uint32_t)(kw * XB + r * 256 + 16 * (c ^ (r & 15)));
  }

  u32x4_t wv[D][4], xv[D][XL];
  // Loads of stage j into ring slot d: x first, so that waiting for a stage's x
  // (the counter retires in order) leaves the younger stages in flight.
  auto issue = [&](int d, int j) __attribute__((always_inline)) {
    const bool on = j < j1;
    const auto xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), 0, on ? x_bytes : 0u, 0x00027000);
    const auto wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.w), 0, on ? w_bytes : 0u, 0x00027000);
    const uint32_t off = (uint32_t)j * (2u * kStageK);
#pragma unroll
    for (int i = 0; i < XL; ++i) xv[d][i] = __builtin_amdgcn_raw_buffer_load_b128(xr, x_off[i] + off, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) wv[d][i] = __builtin_amdgcn_raw_buffer_load_b128(wr, w_off + off + 64 * i, 0, 0);
  };
  f32x4_t acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int d = 0; d < D; ++d) {
    issue(d, j0 + d);
    // Issued in ring order: the waits at the loop's header count on it.
    __builtin_amdgcn_sched_barrier(0);
  }
  auto stage = [&](int d, int b, int j) __attribute__((always_inline)) {
    unsigned char* xb = lds + b * KW * XB;
#pragma unroll
    for (int i = 0; i < XL; ++i)
      if (XALL || x_dst[i] < (uint32_t)((kw + 1) * XB)) *reinterpret_cast<u32x4_t*>(xb + x_dst[i]) = xv[d][i];
    // With RW = 1 the slab's buffer is the wave's own. Otherwise one barrier per
    // stage: a buffer is written again two stages later, after the barrier between.
    if constexpr (RW > 1) __syncthreads();
    else asm volatile("" ::: "memory");
    const unsigned char* xs = xb + kw * XB;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint4 wc = __builtin_bit_cast(uint4, wv[d][i]);
#pragma unroll
      for (int t = 0; t < MT; ++t)
        acc[t] = mfma_16x16x32(wc, ld16(xs + (16 * t + n) * 256 + 16 * ((4 * i + g) ^ n)), acc[t]);
    }
    issue(d, j + D);
  };
  constexpr int U = (D % 2) ? 2 * D : D;  // ring slot and LDS buffer numbers are constants
  for (int s = 0; s < steps; s += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (s + u >= steps) goto summed;
      stage(u % D, u & 1, j0 + s + u);
    }
  }
summed:
  __syncthreads();  // every x read done: the buffers become the exchange of partial sums
  f32x4_t* red = reinterpret_cast<f32x4_t*>(lds);
#pragma unroll
  for (int t = 0; t < MT; ++t) red[(w * MT + t) * 64 + lane] = acc[t];
  __syncthreads();
  for (int it = threadIdx.x; it < CW * MT * 64; it += NW * 64) {
    const int l = it & 63, f = it >> 6, r = f / MT, t = f % MT;
    auto sum = [&](int rr) {
      f32x4_t y = red[(rr * MT + t) * 64 + l];
#pragma unroll
      for (int k = 1; k < KW; ++k) y += red[((k * RW + rr) * MT + t) * 64 + l];
      return y;
    };
    // Lane n + 16g of a result tile: token 16t + n, columns 4g .. 4g + 3.
    const int mb = 16 * t + (l & 15), m = m0 + mb, c = row0 + 16 * r + 4 * (l >> 4);
    if (mb >= m_here || c >= row1) continue;
    f32x4_t y = sum(r), u = y;
    if constexpr (GLU) u = sum(CW + r);
    if (a.k_splits > 1) {
      const int64_t wn = (GLU ? 2 : 1) * (int64_t)a.n;
      float* dst = a.partials + ((int64_t)ks * a.m + m) * wn + c;
#pragma unroll
      for (int i = 0; i < 4; i += 2)
        if (c + i < row1) {
          *reinterpret_cast<f32x2_t*>(dst + i) = f32x2_t{y[i], y[i + 1]};
          if constexpr (GLU) *reinterpret_cast<f32x2_t*>(dst + a.n + i) = f32x2_t{u[i], u[i + 1]};
        }
      continue;
    }
    if constexpr (GLU) {
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = silu(y[i]) * u[i];
    } else {
      y = add_bias(a, c, row1, y);
    }
    store4(a, m, c, row1, y);
  }
}

// Adds the k splits' partial sums in split order and applies the epilogue:
// one thread per (token, 2 columns).
template <bool GLU>
__global__ __launch_bounds__(256) void linear_reduce_kernel(LinearArgs a) {
  const int64_t it = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int pairs = a.n / 2;
  if (it >= (int64_t)a.m * pairs) return;
  const int m = (int)(it / pairs), c = 2 * (int)(it - (int64_t)m * pairs);
  const int64_t wn = (GLU ? 2 : 1) * (int64_t)a.n, step = (int64_t)a.m * wn;
  const float* p = a.partials + (int64_t)m * wn + c;
  f32x2_t y = {0.f, 0.f}, u = {0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < a.k_splits; ++k) {
    y += *reinterpret_cast<const f32x2_t*>(p + k * step);
    if constexpr (GLU) u += *reinterpret_cast<const f32x2_t*>(p + k * step + a.n);
  }
  if constexpr (GLU) {
    y[0] = silu(y[0]) * u[0];
    y[1] = silu(y[1]) * u[1];
  } else if (a.bias != nullptr) {
    const uint16_t* b = reinterpret_cast<const uint16_t*>(a.bias) + c;
    y[0] += bf16_to_f32(b[0]);
    y[1] += bf16_to_f32(b[1]);
  }
  *reinterpret_cast<uint32_t*>(reinterpret_cast<uint16_t*>(a.out) + (int64_t)m * a.out_stride + c) =
      pack_bf16x2_hw(y[0], y[1]);
}

template <int MT, int RW, int KW, int D, bool GLU>
hipError_t launch_tiles(const LinearArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((skinny_linear_kernel<MT, RW, KW, D, GLU>), dim3((unsigned)(a.row_groups * a.k_splits), (unsigned)((a.m + MT * 16 - 1) / (MT * 16))),
                     dim3(RW * KW * 64), 0, s, a);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess || a.k_splits == 1) return err;
  const int64_t items = (int64_t)a.m * (a.n / 2);
  hipLaunchKernelGGL((linear_reduce_kernel<GLU>), dim3((unsigned)((items + 255) / 256)), dim3(256), 0, s, a);
  return hipGetLastError();
}

template <int RW, int KW, int D, bool GLU>
hipError_t launch_waves(const LinearArgs& a, hipStream_t s) {
  if (a.m <= 16) return launch_tiles<1, RW, KW, D, GLU>(a, s);
  if (a.m <= 32) return launch_tiles<2, RW, KW, D, GLU>(a, s);
  if constexpr (RW == 8) {  // beyond 64 tokens (linear_plan): blocks of at most 128, evenly
    const int per_block = (a.m + (a.m + 127) / 128 - 1) / ((a.m + 127) / 128);
    if (per_block > 96) return launch_tiles<8, RW, KW, D, GLU>(a, s);
    if (per_block > 64) return launch_tiles<6, RW, KW, D, GLU>(a, s);
  }
  return launch_tiles<4, RW, KW, D, GLU>(a, s);
}

}  // namespace

// Whether the kernel's call ends sooner than the library's, for n = 16 * tiles columns and
// k = 128 * stages. Measured in graphs of back-to-back calls, weights from HBM, at 7,900 points:
// 640 to 256000 columns, k 384 to 28672, 1 to 256 tokens, and checked at 10,700 random ones (64
// columns and k 128 up), 97% of which are faster and 0.6% more than a twentieth slower (3 of
// them more than a tenth). The library's time jumps with its own choice of tiles, so
// its good shapes lie between bad ones; where they do, the line leaves both to it. Lines and
// figures (us, kernel / library):
//   gated (the library's side includes its SiLU·mul launch): the kernel reads gate and up once
//     and writes half the columns. Lost to a long k with few columns, where a work-group's walk
//     sets the time: 1024 columns, 48 stages, 1 token 16.2 / 14.1; 2048 columns, 33
//     tokens, 28 stages 17.5 / 15.0, 12 stages 9.8 / 12.1. Beyond 64 tokens to all but a short k
//     (2·4864 x 896: 65 tokens 11.1 / 14.2, 128: 14.1 / 15.0, 192: 17.3 / 16.8; 18944 columns, 7
//     stages, 128 tokens 31.1 / 27.2);
//   beyond 17 thousand k the library reads the weights at 1.1 to 1.4 TB/s (3584 x 18944: 16
//     tokens 29 / 46, 64: 36 / 90, 256: 83 / 126; 4096 x 16384, 1 token 35.2 / 33.9, 17408 33.7 / 50.4);
//   a k of 128 beyond 256 columns is two launches' latency either way (2680 columns, 6 tokens 4.0 /
//     3.5);
//   1 to 16 tokens: few rows are the kernel's at any k (16 tokens, 1152 x 896 4.7 / 6.8, 896 x
//     8192 10.1 / 12.2); 160 to 255 tiles up to 35 stages (3584 x 4608 13.1 / 11.4, 4352 12.8 /
//     17.1), 256 to 511 up to 51 (4096 x 6656 17.9 / 15.5), more columns up to 39 (12288 x 5120
//     35.2 / 29.9);
//   17 to 32: 160 to 255 tiles lose from 40 stages (32 tokens, 3584 x 5120 17.0 / 15.8), 288 to
//     320 nowhere (4608 x 3584 0.95 times), the rest of 256 to 511 from 28 or 18 (4096 x 3840
//     14.4 / 13.0, 7168 x 2304 11.7 / 11.2), more columns from 9 (10240 x 1280 12.4 / 10.9), 1024
//     tiles and more at once (17032 x 640, 23 tokens 13.6 / 11.5, 28672 x 896 21.3 / 15.8);
//   33 to 64: x outweighs the weights of few rows per work-group. Below 160 tiles the lines
//     follow the library's jumps (2048 x 2560, 33 tokens 11.1 / 9.3, 1280 x 5632, 48: 12.8 / 10.6,
//     92 x 1792, 33: 8.6 / 7.3, 896 x 896 0.77 times, 896 x 4864 0.70); 256 to 287 tiles up to 20
//     stages (4096 x 3072, 48 tokens 14.7 / 11.4), 288 to 511 up to 29 (4608 x 3584 0.89 times;
//     4608 x 4096, 48 tokens 18.3 / 22.7, 64: 19.4 / 17.8), none beyond (12288 x 3584, 33 tokens
//     32.6 / 23.1);
//   65 to 128: below 192 tiles from 80 or 56 stages (896 x 8192, 65 tokens 14.8 / 13.3; 2560 x
//     6656 18.8 / 19.1), 192 to 320 tiles but for 32 to 43 or 47 (5120 x 4096, 65 tokens 19.7 /
//     17.2, 5632 23.7 / 23.0, 3148 x 4864, 119: 22.6 / 19.8; 3584 x 3584 0.95 times, 4608 x 3584
//     1.01), up to 511 from 64;
//   heads (2048 tiles and more) are within a tenth of each other but for the library's bad
//     sizes (100352 x 896, 17 tokens 42 / 126; 152064 x 3584, 16 tokens 188 / 231): below 32
//     stages, up to 16 tokens; from 4096 tiles up to 32, and to 64 for at most 8 stages (50304 x 896, 48
//     tokens 26.8 / 23.7). 256000 columns are the library's.
// eager: the caller launches call by call. Beyond 64 tokens, where such steps are too large for
// a captured graph, a library GEMM costs it 18 to 24 us of host time and the SiLU·mul 4.5, a call
// here 5 to 8: a kernel that ends within the library's host time is waited for no longer than the
// library's caller would wait for itself. Gated: at most 26 us (MLP 896 x 4864, whole, on two
// hosts: 192 tokens 40 and 53 us with the library, 28 and 32 with the gated kernel, 17.3 / 16.8 on
// the GPU; 256: 40 and 53, 35 and 47; 24.1 / 18.8). Plain: at most 15.5 us (the MLP's 896 x 4864 as
// well: 65 tokens 23.4 and 29.8 -> 21.7 and 23.1, 96: 23.4 and 29.6 -> 22.5 and 24.1, 128 either
// way: 23.5 and 29.6, 26.3 and 28.3).
static bool ends_sooner(int m, int tiles, int stages, bool gated, bool eager, double products) {
  if (gated) {
    if (m <= 16) return stages < 36 || (tiles >= 224 && stages < 64);
    if (m <= 32) return stages < 36 || (tiles >= 352 && stages < 64);
    if (m <= 64) return stages < 18 || (tiles >= 176 && stages < 36) || (tiles >= 560 && stages < 64);
    if (m <= 128 && tiles < 1100 && (stages <= 4 || (tiles >= 64 && stages <= 8) || (tiles >= 300 && stages <= 12)))
      return true;
    return eager && stages <= (m <= 128 ? 12 : 8) && products <= 2.4e9;
  }
  if (stages < 2 && tiles > 16 && tiles < 2048) return false;
  if (tiles >= 2048)
    return m <= 64 && stages < 32 && tiles <= 12800 && (m <= 16 || (tiles >= 4096 && (m <= 32 || stages <= 8)));
  if (stages >= 136 && tiles < 512) return true;
  if (m <= 16) return tiles < 160 || stages < (tiles < 256 ? 36 : tiles < 512 ? 52 : 40);
  if (m <= 32) {
    if (tiles < 160) return stages < 44 || stages >= 52;
    if (tiles < 256) return stages < 40 || stages >= 64;
    if (tiles >= 288 && tiles <= 320) return true;
    if (tiles >= 512) return tiles < 1024 && stages >= 3 && stages < 9;
    return stages < (tiles < 288 ? 28 : 18);
  }
  if (m <= 64) {
    if (tiles < 512 && stages > 64) return true;
    if (tiles < 160)
      return (stages >= 6 && stages <= 8) || (tiles >= 40 && stages >= 12 && stages <= 16) ||
             (stages >= 32 && stages <= (tiles < 96 ? 40 : 63));
    if (tiles < 256) return false;
    if (tiles < 288) return stages <= 20;
    return tiles < 512 && (stages < 30 || (tiles <= 320 && m <= 48));
  }
  if (eager && tiles <= 320 && stages >= 28 && stages < 64 && products <= 4.5e8) return true;
  if (m <= 128) {
    if (tiles < 192) return stages >= (tiles < 160 ? 80 : 56);
    return tiles < 512 &&
           (stages >= 64 || (tiles <= 320 && ((stages >= 28 && stages < 32) || stages >= (tiles < 256 ? 48 : 44))));
  }
  return false;
}

// The launch of a shape, or rw = 0 where the library's GEMM is the better one (ends_sooner; or
// the shape does not fit the kernel). 16-row tiles of weights and 128-wide stages of k decide:
//   gated: 8 row waves beyond 8192 columns, else 4 x 2 (8192 x 2048, 17 tokens 20.3 us on 8, 18.2
//     on 4 x 2: 256 work-groups fill their 32 columns exactly); past 64 tokens 8 row waves in
//     blocks of 65 to 128 tokens;
//   many tiles (>= 2048, a head): 8 row waves, each x stage shared by 128 rows;
//   beyond 64 tokens below 64 stages: 8 x 1 with k cut by 3 stages or more until tiles x splits
//     reach 1536;
//   long k (>= 64 stages, or >= 32 with few rows and more than 16 tokens): 4 row waves x 2
//     slabs, k cut over work-groups until tiles x splits reach about 1000 (past 32 tokens and 64
//     stages 8 x 1, twice the splits, in blocks of at most 128 tokens);
//   the rest: 2 x 4 from 160 tiles, 1 x 4 below (each work-group then streams a
//     few rows with 4 waves and no sum across work-groups).
LinearPlan linear_plan(int32_t m, int32_t n, int32_t k, bool gated, bool eager) {
  LinearPlan p{};
  const int64_t rows = (gated ? 2 : 1) * (int64_t)n;
  if (m < 1 || m > 256 || n < 64 || n % 4 != 0 || k < kStageK || k % kStageK != 0) return p;
  if (rows * k * 2 >= (int64_t)kNoLoad) return p;
  const int tiles = (n + 15) / 16, stages = k / kStageK;
  if (!ends_sooner(m, tiles, stages, gated, eager, (double)m * rows * k)) return p;
  p.k_splits = 1;
  if (gated) {
    p.rw = n > 8192 || m > 64 ? 8 : 4;
  } else if (tiles >= 2048) {
    p.rw = 8;
  } else if (m > 64 && stages < 64) {
    p.rw = 8;
    p.k_splits = std::max(1, std::min(stages / 3, 1536 / tiles));
  } else if (stages >= 64 || (stages >= 32 && tiles < 160 && m > 16)) {
    const bool wide = m > 32 && stages >= 64;
    p.rw = wide ? 8 : 4;
    p.k_splits = std::max(1, std::min(stages / 4, ((wide ? 2048 : 1024) - 1) / tiles));
  } else {
    p.rw = tiles >= 160 ? 2 : 1;
  }
  p.kw = p.rw == 1 ? 4 : 8 / p.rw;
  const int cols = 16 * (gated ? p.rw / 2 : p.rw);
  const int groups = (n + cols - 1) / cols;
  const int cus = device_cus();
  p.row_groups = (groups * p.k_splits + cus - 1) / cus * cus / p.k_splits;
  p.unit = n / p.row_groups >= 64 ? 4 : 2;
  p.row_groups = std::max(groups, std::min(p.row_groups, n / p.unit));
  // An even split in units may exceed a work-group's tiles by a unit.
  while (((int64_t)(n / p.unit) + p.row_groups - 1) / p.row_groups * p.unit > cols) ++p.row_groups;
  p.partial_bytes = p.k_splits > 1 ? (int64_t)p.k_splits * m * rows * 4 : 0;
  return p;
}

hipError_t skinny_linear(const LinearArgs& args, bool gated, bool eager, hipStream_t s) {
  LinearArgs a = args;
  const LinearPlan p = linear_plan(a.m, a.n, a.k, gated, eager);
  if (p.rw == 0 || (int64_t)a.m * a.x_stride * 2 >= (int64_t)kNoLoad) return hipErrorInvalidValue;
  if (p.k_splits > 1 && a.partials == nullptr) return hipErrorInvalidValue;
  a.k_splits = p.k_splits;
  a.row_groups = p.row_groups;
  a.unit = p.unit;
  if (gated) return p.rw == 8 ? launch_waves<8, 1, 2, true>(a, s) : launch_waves<4, 2, 2, true>(a, s);
  switch (p.rw) {
    case 8: return launch_waves<8, 1, 2, false>(a, s);
    case 4: return launch_waves<4, 2, 2, false>(a, s);
    case 2: return launch_waves<2, 4, 2, false>(a, s);
    default: return launch_waves<1, 4, 3, false>(a, s);
  }
}

}  // namespace bvllm
