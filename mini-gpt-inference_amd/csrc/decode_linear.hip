// decode_linear.hip -- the linear layers of a decode step for gfx950, up to
// kLinearMaxRows rows (one token per sequence), bf16 and f16:
//   mgi_decode_linear       out = act(x W^T + bias)             one launch
//   mgi_decode_linear_norm  out = x W^T + bias + residual, norm = LN(out)   two
// They stand for the PyTorch calls around the attention of a transformer block
// (minivllm/block.py:72-93: linear, linear -> gelu, linear -> add -> layer_norm)
// and before the LM head (minivllm/model.py:218-248).
//
// At these row counts each layer is bound by reading its weights once (6.15
// TB/s here past the first microseconds) and by what every launch costs
// before that (2.2 us, and 2-3 us until its loads stream), so the elementwise
// neighbours ride along: bias and GELU in the sums' epilogue, residual and
// LayerNorm in the pass that adds the K splits.
#include "mgi_common.h"
#include "mgi_internal.h"
#include "minivllm_hip.h"

namespace mgi {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <typename T> struct Mma;
template <> struct Mma<bf16_t> {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  typedef __bf16 v2 __attribute__((ext_vector_type(2)));
  __device__ static __forceinline__ f32x4_t mfma(uint4 a, uint4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
  }
  __device__ static __forceinline__ uint32_t pack2(float lo, float hi) {
    const v2 v = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, v);
  }
  __device__ static __forceinline__ float lo(uint32_t w) { return bf16_lo(w); }
  __device__ static __forceinline__ float hi(uint32_t w) { return bf16_hi(w); }
};
template <> struct Mma<f16_t> {
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  typedef _Float16 v2 __attribute__((ext_vector_type(2)));
  __device__ static __forceinline__ f32x4_t mfma(uint4 a, uint4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
  }
  __device__ static __forceinline__ uint32_t pack2(float lo, float hi) {
    const v2 v = {(_Float16)lo, (_Float16)hi};
    return __builtin_bit_cast(uint32_t, v);
  }
  __device__ static __forceinline__ float lo(uint32_t w) { return f16_to_f32((uint16_t)(w & 0xffffu)); }
  __device__ static __forceinline__ float hi(uint32_t w) { return f16_to_f32((uint16_t)(w >> 16)); }
};

constexpr int kWaves = 8;    // wavefronts per workgroup; they split K
constexpr int kUnit = 64;    // k values of one unit: a 128-byte line of a weight row
constexpr int kTileN = 16;   // output columns (weight rows) per tile

// Weight tiles a wavefront of the resident kernel has in flight: as many as its
// 256 registers hold beside x.
constexpr int weight_tiles(int MT, int U) { return 8 * U * (MT + 2) <= 200 ? 2 : 1; }

// Joins the workgroup after this wavefront's LDS accesses; loads in flight
// stay in flight (a __syncthreads would drain the next tile's weights).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <typename T>
__device__ __forceinline__ uint4 load16(const T* p) { return *reinterpret_cast<const uint4*>(p); }

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.f + erff(x * 0.70710678118654752f)); }

// Epilogue of one 16-column tile: thread (mt, lane) adds the eight
// wavefronts' partial sums of row 16 mt + lane % 16, columns n0 + 4 (lane /
// 16) .. + 3, in wavefront order, and stores them.
template <typename T, int MT>
__device__ __forceinline__ void finish_tile(const LinearArgs& a, const float4 (&red)[kWaves][MT][64], int n0) {
  using MM = Mma<T>;
  const int mt = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
  if (mt >= MT) return;
  const int row = 16 * mt + (lane & 15), n = n0 + 4 * (lane >> 4);
  if (row >= a.B || n >= a.N) return;
  const T* bias = reinterpret_cast<const T*>(a.bias);
  T* out = reinterpret_cast<T*>(a.out) + (int64_t)row * a.N + n;
  float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const float4 p = red[w][mt][lane];
    s[0] += p.x;
    s[1] += p.y;
    s[2] += p.z;
    s[3] += p.w;
  }
  if ((a.N & 3) == 0) {  // rows of 8-byte aligned groups of four
    uint2 b2 = make_uint2(0u, 0u);
    if (bias) b2 = *reinterpret_cast<const uint2*>(bias + n);
    s[0] += MM::lo(b2.x);
    s[1] += MM::hi(b2.x);
    s[2] += MM::lo(b2.y);
    s[3] += MM::hi(b2.y);
    if (a.gelu) {
#pragma unroll
      for (int i = 0; i < 4; ++i) s[i] = gelu(s[i]);
    }
    *reinterpret_cast<uint2*>(out) = make_uint2(MM::pack2(s[0], s[1]), MM::pack2(s[2], s[3]));
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (n + i >= a.N) break;
      float x = s[i] + (bias ? Elem<T>::load(bias + n + i) : 0.f);
      Elem<T>::store(out + i, a.gelu ? gelu(x) : x);
    }
  }
}

// A workgroup computes 16-column tiles of the output for all rows: its eight
// wavefronts take the 64-wide units of K in turn (unit w + 8 u), so each
// reads whole 128-byte lines of the 16 weight rows and keeps its share of x,
// U units of MT 16-row blocks, in registers as MFMA operands for every tile.
// Products are 16x16x32 (A: 16 weight rows, B: 16 rows of x), so a lane
// holds four columns of one row; the wavefronts' sums meet in LDS.
//
// One workgroup per CU walks the tiles (launching costs about 1 ns per
// wavefront, so two per CU with one tile each were slower: 14.5 against 11.5
// us at 16 x 2048 -> 8192), with the next tiles' weights in flight. Measured on
// MI355X (us; PyTorch's calls / this; bf16, K = 2048): 16 rows to 6144 columns
// 12.9 / 10.2, to 8192 with GELU 17.5 / 11.5, to 32000 33.5 / 27.8 (4.7 TB/s of
// weights); 40 rows 13.6 / 13.5 and 18.3 / 15.1; 64 rows, K = 512, to 1536
// 7.3 / 4.7. What grows with the rows is x, which every workgroup reads whole
// through one CU's 40-70 KB/us. Weights read non-temporally were 5-10 % slower:
// an operand load touches half a line of 16 rows, and the other half then comes
// from memory again. Splitting K here too (2-8 ways, sums added by a second
// launch) lost 5-60 %.
template <typename T, int MT, int U>
__global__ void __launch_bounds__(64 * kWaves, 2) decode_linear_resident(const LinearArgs a) {
  using MM = Mma<T>;
  __shared__ float4 red[2][kWaves][MT][64];
  const int lane = (int)threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int nunits = a.K / kUnit, ntiles = (a.N + kTileN - 1) / kTileN;
  const T* W = reinterpret_cast<const T*>(a.w);

  auto load_w = [&](int tile, uint4 (&wf)[U][2]) {
    const T* row = W + (int64_t)min(tile * kTileN + c, a.N - 1) * a.K + 8 * g;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        wf[u][j] = w + kWaves * u < nunits ? load16(row + (w + kWaves * u) * kUnit + 32 * j)
                                           : make_uint4(0u, 0u, 0u, 0u);
  };
  // Everything the first tiles need goes out at once.
  constexpr int WT = weight_tiles(MT, U);
  uint4 xf[MT][U][2], wf[WT][U][2];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int row = 16 * mt + c;
    const T* x = reinterpret_cast<const T*>(a.x) + (int64_t)min(row, a.B - 1) * a.K + 8 * g;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        xf[mt][u][j] = row < a.B && w + kWaves * u < nunits ? load16(x + (w + kWaves * u) * kUnit + 32 * j)
                                                             : make_uint4(0u, 0u, 0u, 0u);
  }
  const int step = (int)gridDim.x;
  int tile = (int)blockIdx.x;
#pragma unroll
  for (int t = 0; t < WT; ++t)
    if (tile + t * step < ntiles) load_w(tile + t * step, wf[t]);
  __builtin_amdgcn_sched_barrier(0);

  while (true) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {  // two reduction buffers; weight buffer t % WT
      f32x4_t acc[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[mt] = MM::mfma(wf[t % WT][u][j], xf[mt][u][j], acc[mt]);
      const int n0 = tile * kTileN;
      if (tile + WT * step < ntiles) load_w(tile + WT * step, wf[t % WT]);
      tile += step;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) red[t][w][mt][lane] = make_float4(acc[mt][0], acc[mt][1], acc[mt][2], acc[mt][3]);
      // One barrier per tile: the sums of tile i + 2 reuse tile i's buffer after
      // the barrier of tile i + 1, which the threads finishing tile i join later.
      lds_barrier();
      finish_tile<T, MT>(a, red[t], n0);
      if (tile >= ntiles) return;
    }
  }
}

// Wide K, few columns (the projections back to the residual stream): the
// columns alone do not fill the chip, and a workgroup that walked all of K
// would read all of x. A workgroup takes 64 columns (four wavefronts of 16)
// and one of the K splits: its share of x goes to LDS once for the four, its
// weights to registers, everything in flight at once, and its f32 sums to
// part[split][row][column]; decode_reduce adds the splits. Measured on MI355X
// (us; PyTorch's linear, add and layer_norm / both launches; bf16, to 2048
// columns): K = 2048, 16 rows 14.2 / 7.9, 64 rows 14.8 / 10.8; K = 8192, 20.1 /
// 13.8 and 29.3 / 19.0; to 4096 columns (replayed, weights from memory): K = 4096,
// 24.2 / 14.6 and 24.0 / 17.6; K = 16 384, 40.1 / 39.1. More than 32 rows of more
// than 8192 hold one workgroup per CU (128 KiB of x): 40 rows, K = 10 240, to 2560,
// 28.7 / 31.4, K = 16 384, to 4096, 33 rows 45.8 / 62.4 (mgi_decode_linear_norm_pays).
// Walking all of K per workgroup (128 workgroups, residual
// in the epilogue, no second launch) took 17.8 and 38.8 for K = 8192.
constexpr int kSplitWaves = 4;
constexpr int kSplitN = kSplitWaves * kTileN;

template <typename T, int MT, int UK>
__global__ void __launch_bounds__(64 * kSplitWaves, 1) decode_linear_split(const LinearArgs a) {
  using MM = Mma<T>;
  constexpr int ROWB = UK * kUnit * 2;  // bytes per row of the x share
  constexpr int CPR = ROWB / 16;        // 16-byte chunks per row; chunk q of row r is stored at q ^ (r & 7)
  constexpr int XL = 16 * MT * CPR / (64 * kSplitWaves);  // chunks per thread
  __shared__ __align__(16) unsigned char xs[16 * MT * ROWB];
  const int tid = (int)threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = ((int)blockIdx.x * kSplitWaves + w) * kTileN;
  const int u0 = (int)blockIdx.y * a.split_units;              // first unit of this split
  const int nu = min(a.split_units, a.K / kUnit - u0);         // its units (1 .. UK)
  const T* x = reinterpret_cast<const T*>(a.x) + u0 * kUnit;
  const T* wr = reinterpret_cast<const T*>(a.w) + (int64_t)min(n0 + c, a.N - 1) * a.K + u0 * kUnit + 8 * g;
  uint4 xv[XL], wf[UK][2];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int it = tid + 64 * kSplitWaves * i, row = it / CPR, q = it % CPR;
    xv[i] = row < a.B && q < 8 * nu ? load16(x + (int64_t)row * a.K + 8 * q) : make_uint4(0u, 0u, 0u, 0u);
  }
#pragma unroll
  for (int u = 0; u < UK; ++u)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      wf[u][j] = u < nu ? load16(wr + u * kUnit + 32 * j) : make_uint4(0u, 0u, 0u, 0u);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int it = tid + 64 * kSplitWaves * i, row = it / CPR, q = it % CPR;
    *reinterpret_cast<uint4*>(xs + row * ROWB + ((q ^ (row & 7)) << 4)) = xv[i];
  }
  lds_barrier();
  f32x4_t acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < UK; ++u)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int row = 16 * mt + c, q = 8 * u + 4 * j + g;
        acc[mt] = MM::mfma(wf[u][j], *reinterpret_cast<const uint4*>(xs + row * ROWB + ((q ^ (row & 7)) << 4)), acc[mt]);
      }
  const int n = n0 + 4 * g;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int row = 16 * mt + c;
    if (row < a.B && n < a.N)
      *reinterpret_cast<float4*>(a.part + ((int64_t)blockIdx.y * a.B + row) * a.N + n) =
          make_float4(acc[mt][0], acc[mt][1], acc[mt][2], acc[mt][3]);
  }
}

// out = sum of the splits + bias + residual, one workgroup per row, and with
// gamma also norm = LayerNorm(out) of the stored (rounded) row, in two passes
// in f32. With no splits, norm = LayerNorm(residual) alone.
constexpr int kReduceThreads = 512;

__device__ __forceinline__ float block_sum(float x, float* red) {
  x = wave_sum(x);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < kReduceThreads / 64; ++i) t += red[i];
  return t;
}

template <typename T>
__global__ void __launch_bounds__(kReduceThreads) decode_reduce(const LinearArgs a) {
  using MM = Mma<T>;
  constexpr int G = kReduceMaxN / (4 * kReduceThreads);  // 4-column groups per thread
  __shared__ float red[2][kReduceThreads / 64];
  const int row = (int)blockIdx.x;
  const int64_t r0 = (int64_t)row * a.N;
  float s[G][4];
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < G; ++i) {
    const int n = 4 * ((int)threadIdx.x + kReduceThreads * i);
    if (n >= a.N) continue;
    const uint2 rs = *reinterpret_cast<const uint2*>(reinterpret_cast<const T*>(a.res) + r0 + n);
    float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
    const float* p = a.part + r0 + n;
    const int64_t ps = (int64_t)a.B * a.N;
#pragma unroll 8
    for (int k = 0; k < a.splits; ++k) {
      const float4 v = *reinterpret_cast<const float4*>(p + k * ps);
      t.x += v.x;
      t.y += v.y;
      t.z += v.z;
      t.w += v.w;
    }
    uint2 bs = make_uint2(0u, 0u);
    if (a.bias) bs = *reinterpret_cast<const uint2*>(reinterpret_cast<const T*>(a.bias) + n);
    const uint2 o = make_uint2(MM::pack2(t.x + MM::lo(bs.x) + MM::lo(rs.x), t.y + MM::hi(bs.x) + MM::hi(rs.x)),
                               MM::pack2(t.z + MM::lo(bs.y) + MM::lo(rs.y), t.w + MM::hi(bs.y) + MM::hi(rs.y)));
    if (a.out)
      *reinterpret_cast<uint2*>(reinterpret_cast<T*>(a.out) + r0 + n) = o;
    s[i][0] = MM::lo(o.x);
    s[i][1] = MM::hi(o.x);
    s[i][2] = MM::lo(o.y);
    s[i][3] = MM::hi(o.y);
    sum += (s[i][0] + s[i][1]) + (s[i][2] + s[i][3]);
  }
  if (!a.gamma) return;
  const float mean = block_sum(sum, red[0]) / (float)a.N;
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < G; ++i) {
    if (4 * ((int)threadIdx.x + kReduceThreads * i) >= a.N) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s[i][e] -= mean;
      sq = fmaf(s[i][e], s[i][e], sq);
    }
  }
  const float rstd = rsqrtf(block_sum(sq, red[1]) / (float)a.N + a.eps);
#pragma unroll
  for (int i = 0; i < G; ++i) {
    const int n = 4 * ((int)threadIdx.x + kReduceThreads * i);
    if (n >= a.N) continue;
    const uint2 gw = *reinterpret_cast<const uint2*>(reinterpret_cast<const T*>(a.gamma) + n);
    const uint2 bw = *reinterpret_cast<const uint2*>(reinterpret_cast<const T*>(a.beta) + n);
    *reinterpret_cast<uint2*>(reinterpret_cast<T*>(a.norm) + r0 + n) =
        make_uint2(MM::pack2(fmaf(s[i][0] * rstd, MM::lo(gw.x), MM::lo(bw.x)), fmaf(s[i][1] * rstd, MM::hi(gw.x), MM::hi(bw.x))),
                   MM::pack2(fmaf(s[i][2] * rstd, MM::lo(gw.y), MM::lo(bw.y)), fmaf(s[i][3] * rstd, MM::hi(gw.y), MM::hi(bw.y))));
  }
}

template <typename T, int MT, int U>
void launch_resident(const LinearArgs& a, hipStream_t stream) {
  const int ntiles = (a.N + kTileN - 1) / kTileN;
  const dim3 grid((unsigned)(ntiles < a.cus ? ntiles : a.cus)), block(64 * kWaves);
  hipLaunchKernelGGL((decode_linear_resident<T, MT, U>), grid, block, 0, stream, a);
}

template <typename T, int MT>
hipError_t launch_mt(const LinearArgs& a, hipStream_t stream) {
  switch ((a.K + kWaves * kUnit - 1) / (kWaves * kUnit)) {
    case 1: launch_resident<T, MT, 1>(a, stream); break;
    case 2: launch_resident<T, MT, 2>(a, stream); break;
    case 3: launch_resident<T, MT, 3>(a, stream); break;
    case 4: launch_resident<T, MT, 4>(a, stream); break;
    case 5: launch_resident<T, MT, 5>(a, stream); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <typename T>
hipError_t launch_t(const LinearArgs& a, hipStream_t stream) {
  if (a.B <= 16) return launch_mt<T, 1>(a, stream);
  if (a.B <= 32) return launch_mt<T, 2>(a, stream);
  return launch_mt<T, 4>(a, stream);
}

template <typename T, int MT>
void launch_split_mt(const LinearArgs& a, hipStream_t stream) {
  const dim3 grid((unsigned)((a.N + kSplitN - 1) / kSplitN), (unsigned)a.splits), block(64 * kSplitWaves);
#define MGI_SPLIT(UK) hipLaunchKernelGGL((decode_linear_split<T, MT, UK>), grid, block, 0, stream, a)
  if (a.split_units <= 2) MGI_SPLIT(2);
  else if (a.split_units <= 4) MGI_SPLIT(4);
  else if (a.split_units <= 8) MGI_SPLIT(8);
  else if (a.split_units <= 12) MGI_SPLIT(12);
  else MGI_SPLIT(16);
#undef MGI_SPLIT
}

template <typename T>
hipError_t launch_split_t(const LinearArgs& a, hipStream_t stream) {
  if (a.splits > 0) {
    if (a.B <= 16) launch_split_mt<T, 1>(a, stream);
    else if (a.B <= 32) launch_split_mt<T, 2>(a, stream);
    else launch_split_mt<T, 4>(a, stream);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((decode_reduce<T>), dim3((unsigned)a.B), dim3(kReduceThreads), 0, stream, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_decode_linear(const LinearArgs& a, int dtype, hipStream_t stream) {
  return dtype == MGI_BF16 ? launch_t<bf16_t>(a, stream) : launch_t<f16_t>(a, stream);
}

hipError_t launch_decode_linear_split(const LinearArgs& a, int dtype, hipStream_t stream) {
  return dtype == MGI_BF16 ? launch_split_t<bf16_t>(a, stream) : launch_split_t<f16_t>(a, stream);
}

}  // namespace mgi
