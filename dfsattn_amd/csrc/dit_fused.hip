// Fused elementwise kernels of the DiT block around the attention (the Wan
// transformer block of diffusers that the reference's Wan driver loads,
// wan21_t2v_inference.py:102-103): the fp32 LayerNorm with adaLN modulation,
//   y = bf16((LN(x) [* w + b]) * (1 + scale) + shift),
// and the gated residual,
//   out = bf16(float(x) + float(y) * gate),
// each one pass over the rows instead of torch's chain of dtype copies and
// broadcast ops. Every fp32 product and sum is rounded separately, in the
// order torch evaluates the same expressions; only the LayerNorm's reduction
// order differs.
#include "common.h"

namespace dfs {
namespace {

constexpr int kMaxChunks = 16;  // at most 16 x 512 channels per row

template <bool F16>
__device__ __forceinline__ float to_f32(uint32_t bits) {
  return F16 ? f16_bits_to_f32(bits) : bf16_bits_to_f32(bits);
}

template <bool F16>
__device__ __forceinline__ uint32_t from_f32(float v) {
  return F16 ? f32_to_f16_bits(v) : f32_to_bf16_bits(v);
}

template <int CTRL>
__device__ __forceinline__ float dpp_plus(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}

// Sum over the wave, the same bits in every lane: each step adds a value and
// its mirror (or the other half's), so both sides form the same sum. Register
// moves throughout; through LDS (__shfl_xor) the two reductions of a row were
// the longest part of its chain.
__device__ __forceinline__ float wave_sum(float v) {
  v = dpp_plus<0xB1>(v);   // quad_perm [1, 0, 3, 2]
  v = dpp_plus<0x4E>(v);   // quad_perm [2, 3, 0, 1]
  v = dpp_plus<0x141>(v);  // row_half_mirror: the other four lanes of eight
  v = dpp_plus<0x140>(v);  // row_mirror: the other eight of sixteen
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

__device__ __forceinline__ void load8(const float* p, float* v) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  const float4 b = *reinterpret_cast<const float4*>(p + 4);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
  v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

// One wave per RPW rows of C channels (16-byte chunks, 512 channels per wave
// step, the rows held in registers for the two-pass mean and variance).
// HBM-bound (one read and one write of x; a device copy of the same bytes
// takes 125 us at 32,760 x 5,120). The fp32 vectors come from L2 for every
// wave, 4 bytes a channel and vector beside a row's own 2, so large calls give
// a wave two rows per fetch: 140 us against 158 with one row and 211 with the
// types chosen at run time and the reductions through LDS. A workgroup per row
// with the vectors kept in registers took 208 us (two barriers per row).
template <int NCH, bool F16, int RPW>
__global__ void __launch_bounds__(256) adaln_kernel(const uint16_t* __restrict__ x, int64_t rows, int C,
                                                    const float* __restrict__ weight, const float* __restrict__ bias,
                                                    const float* __restrict__ scale, const float* __restrict__ shift,
                                                    float eps, uint16_t* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6)) * RPW;
  if (row >= rows) return;
  const int n = rows - row < RPW ? 1 : RPW;  // rows of this wave; a missing second row repeats the first
  const uint16_t* xr = x + row * C;
  uint4 v[RPW][NCH];
#pragma unroll
  for (int q = 0; q < RPW; ++q)
#pragma unroll
    for (int j = 0; j < NCH; ++j) {
      const int e = j * 512 + lane * 8;
      v[q][j] = make_uint4(0, 0, 0, 0);
      if (e < C) v[q][j] = load_stream(reinterpret_cast<const uint4*>(xr + (q < n ? q : 0) * static_cast<int64_t>(C) + e));
    }
  float mean[RPW], rstd[RPW];
#pragma unroll
  for (int q = 0; q < RPW; ++q) {
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < NCH; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i) sum += to_f32<F16>(u16_at(v[q][j], i));  // zeros past the row's end
    mean[q] = wave_sum(sum) / static_cast<float>(C);
  }
#pragma unroll
  for (int q = 0; q < RPW; ++q) {
    float sq = 0.f;
#pragma unroll
    for (int j = 0; j < NCH; ++j) {
      if (j * 512 + lane * 8 < C) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float d = to_f32<F16>(u16_at(v[q][j], i)) - mean[q];
          sq += d * d;
        }
      }
    }
    rstd[q] = 1.0f / sqrtf(wave_sum(sq) / static_cast<float>(C) + eps);
  }
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int e = j * 512 + lane * 8;
    if (e >= C) continue;
    float w[8], b[8], sc[8], sh[8];
    if (weight) load8(weight + e, w);
    if (bias) load8(bias + e, b);
    if (scale) load8(scale + e, sc);
    if (shift) load8(shift + e, sh);
#pragma unroll
    for (int q = 0; q < RPW; ++q) {
      if (q >= n) continue;
      uint32_t packed[4];
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        float y2[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma clang fp contract(off)
          float y = (to_f32<F16>(u16_at(v[q][j], i + t)) - mean[q]) * rstd[q];
          if (weight) y = y * w[i + t];
          if (bias) y = y + b[i + t];
          if (scale) y = y * (1.0f + sc[i + t]);
          if (shift) y = y + sh[i + t];
          y2[t] = y;
        }
        packed[i / 2] = from_f32<F16>(y2[0]) | (from_f32<F16>(y2[1]) << 16);
      }
      store_stream(reinterpret_cast<uint4*>(out + (row + q) * C + e),
                   make_uint4(packed[0], packed[1], packed[2], packed[3]));
    }
  }
}

struct AdalnArgs {
  const uint16_t* x;
  int64_t rows;
  int C;
  const float *weight, *bias, *scale, *shift;
  float eps;
  uint16_t* out;
};

template <int NCH, int RPW>
void launch_adaln_as(const AdalnArgs& a, bool f16, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>((a.rows + 4 * RPW - 1) / (4 * RPW)));
  if (f16)
    adaln_kernel<NCH, true, RPW><<<grid, 256, 0, s>>>(a.x, a.rows, a.C, a.weight, a.bias, a.scale, a.shift, a.eps, a.out);
  else
    adaln_kernel<NCH, false, RPW><<<grid, 256, 0, s>>>(a.x, a.rows, a.C, a.weight, a.bias, a.scale, a.shift, a.eps, a.out);
}

// Two rows per wave from 8,192 rows on, where the halved wave count still
// gives each of the 1,024 SIMDs four waves, and while two rows fit the
// registers (20 chunks of 16 bytes: 218 VGPRs at 5,120 channels).
template <int NCH>
void launch_adaln(const AdalnArgs& a, bool f16, hipStream_t s) {
  if constexpr (NCH <= 10) {
    if (a.rows >= 8192) return launch_adaln_as<NCH, 2>(a, f16, s);
  }
  launch_adaln_as<NCH, 1>(a, f16, s);
}

// out = float(x) + float(y) * gate[c], eight channels per thread. HBM-bound:
// streaming accesses and one conversion per type reach 6.4 TB/s (158 us at
// 32,760 x 5,120; 174 us with ordinary accesses and run-time types).
// STREAM: for tensors beyond the last-level cache. Below it they take longer
// than ordinary accesses where x and y were just written (8,000 x 5,120: 38.3
// against 35.2 us; 4,000: 19.9, 18.0) and as long where they were not (40.3,
// 39.1); above, 10,000 x 5,120: 48.1 against 52.1 and 49.8 against 51.2.
// x and out may alias (each thread reads its eight elements before writing them).
template <bool F16, bool STREAM>
__global__ void __launch_bounds__(256) gated_residual_kernel(const uint16_t* x, const uint16_t* __restrict__ y,
                                                             const float* __restrict__ gate, int64_t n8, int C,
                                                             uint16_t* out) {
  const int64_t i8 = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i8 >= n8) return;
  const int64_t e = i8 * 8;
  const uint4 xv = load_chunk<STREAM>(reinterpret_cast<const uint4*>(x + e));
  const uint4 yv = load_chunk<STREAM>(reinterpret_cast<const uint4*>(y + e));
  const int c = static_cast<int>(e % C);
  float g[8];
  load8(gate + c, g);
  uint32_t packed[4];
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    float r[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma clang fp contract(off)
      r[t] = to_f32<F16>(u16_at(xv, i + t)) + to_f32<F16>(u16_at(yv, i + t)) * g[i + t];
    }
    packed[i / 2] = from_f32<F16>(r[0]) | (from_f32<F16>(r[1]) << 16);
  }
  store_chunk<STREAM>(reinterpret_cast<uint4*>(out + e), make_uint4(packed[0], packed[1], packed[2], packed[3]));
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace
}  // namespace dfs

extern "C" int dfs_adaln_modulate(const void* x, int64_t rows, int64_t channels, int dtype, const float* weight,
                                  const float* bias, const float* scale, const float* shift, float eps, void* out,
                                  dfs_stream_t stream) {
  using namespace dfs;
  const char* name = "adaln_modulate";
  DFS_REQUIRE(x && out, "%s: x and out must be non-NULL", name);
  DFS_REQUIRE(rows > 0 && channels > 0 && channels % 8 == 0 && channels <= 512 * kMaxChunks,
              "%s: channels=%lld must be a positive multiple of 8 up to %d", name, (long long)channels,
              512 * kMaxChunks);
  DFS_REQUIRE(dtype == DFS_DTYPE_BF16 || dtype == DFS_DTYPE_F16, "%s: dtype must be bf16 or f16", name);
  DFS_REQUIRE(eps >= 0.f, "%s: eps must be non-negative", name);
  const void* ptrs[6] = {x, out, weight, bias, scale, shift};
  for (const void* q : ptrs) DFS_REQUIRE(q == nullptr || aligned16(q), "%s: operands must be 16-byte aligned", name);
  DFS_REQUIRE((rows + 3) / 4 < (int64_t(1) << 31), "%s: too many rows", name);
  const int nch = static_cast<int>((channels + 511) / 512);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const AdalnArgs a{static_cast<const uint16_t*>(x), rows, static_cast<int>(channels), weight, bias, scale, shift, eps,
                    static_cast<uint16_t*>(out)};
  const bool f16 = dtype == DFS_DTYPE_F16;
  switch ((nch + 1) / 2) {  // smallest even chunk count that covers the row
    case 1: launch_adaln<2>(a, f16, st); break;
    case 2: launch_adaln<4>(a, f16, st); break;
    case 3: launch_adaln<6>(a, f16, st); break;
    case 4: launch_adaln<8>(a, f16, st); break;
    case 5: launch_adaln<10>(a, f16, st); break;
    case 6: launch_adaln<12>(a, f16, st); break;
    case 7: launch_adaln<14>(a, f16, st); break;
    case 8: launch_adaln<16>(a, f16, st); break;
    default:
      set_error("%s: internal chunk count %d", name, nch);
      return 1;
  }
  return check_launch(name);
}

extern "C" int dfs_gated_residual(const void* x, const void* y, const float* gate, int64_t rows, int64_t channels,
                                  int dtype, void* out, dfs_stream_t stream) {
  using namespace dfs;
  const char* name = "gated_residual";
  DFS_REQUIRE(x && y && gate && out, "%s: NULL operand", name);
  DFS_REQUIRE(rows > 0 && channels > 0 && channels % 8 == 0, "%s: channels=%lld must be a positive multiple of 8",
              name, (long long)channels);
  DFS_REQUIRE(dtype == DFS_DTYPE_BF16 || dtype == DFS_DTYPE_F16, "%s: dtype must be bf16 or f16", name);
  DFS_REQUIRE(aligned16(x) && aligned16(y) && aligned16(gate) && aligned16(out),
              "%s: operands must be 16-byte aligned", name);
  DFS_REQUIRE(channels < (int64_t(1) << 31), "%s: too many channels", name);
  const int64_t n8 = rows * channels / 8;
  const int64_t blocks = (n8 + 255) / 256;
  DFS_REQUIRE(blocks < (int64_t(1) << 31), "%s: too many elements", name);
  const dim3 grid(static_cast<unsigned>(blocks)), block(256);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const uint16_t *xp = static_cast<const uint16_t*>(x), *yp = static_cast<const uint16_t*>(y);
  uint16_t* op = static_cast<uint16_t*>(out);
  const bool f16 = dtype == DFS_DTYPE_F16, stream_data = n8 * 16 * 3 > kLastLevelCache;
  auto run = [&](auto kernel) { kernel<<<grid, block, 0, st>>>(xp, yp, gate, n8, static_cast<int>(channels), op); };
  if (stream_data)
    f16 ? run(gated_residual_kernel<true, true>) : run(gated_residual_kernel<false, true>);
  else
    f16 ? run(gated_residual_kernel<true, false>) : run(gated_residual_kernel<false, false>);
  return check_launch(name);
}
