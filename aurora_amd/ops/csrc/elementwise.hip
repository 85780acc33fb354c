// Fused element-wise / normalisation kernels (bf16, gfx950).
//
// All memory-bound: bf16 loads vectorized as shortx8 (16 B/lane), grid-stride,
// fused passes so a tensor is read exactly once. The engine's per-layer hot path,
// without an analog in the reference.
#include <type_traits>

#include "common.h"
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

#define CUR_STREAM c10::hip::getCurrentHIPStream().stream()

// ---------------------------------------------------------------- rmsnorm

// Eight results of a product in parts, each rounded to bf16 as the product would be
DEVINL void add_parts8(float (&y)[8], const float* x, int parts, long step) {
#pragma unroll
  for (int j = 0; j < 8; ++j) y[j] = 0.f;
#pragma unroll 4
  for (int p = 0; p < parts; ++p) {
    const floatx4 a = *reinterpret_cast<const floatx4*>(x + p * step);
    const floatx4 b = *reinterpret_cast<const floatx4*>(x + p * step + 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      y[j] += a[j];
      y[4 + j] += b[j];
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) y[j] = bf16_to_f32(f32_to_bf16(y[j]));
}


// One workgroup per row; 256 threads; row length H must be a multiple of 8.
// RESIDUAL: also adds `res` first and writes the sum back to res_out.
// PARTS: x is the sum, rounded to bf16, of `parts` fp32 terms that lie `step` apart. A
// product left in parts is so added up where it is read anyway: 23 rows of 2048 in 8 parts
// 3.8 us, 96 rows of 4096 in 4 parts 4.4; a kernel to add the parts takes 2.4 to 4.7 more.
// N: vectors of eight that a thread holds, so that a row is read once and the weight comes with
// it; 0 for rows too long for that, which are read again. Read again, and held: 6176 rows of
// 4096 42.6 and 34.5 us (5.9 TB/s, the bound), 1600 12.7 and 11.9, one row in 4 parts 3.25 and
// 2.99 (a launch and two trips to memory), 23 of 2048 in 8 parts 4.07 and 3.80.
template <bool RESIDUAL, bool PARTS, int N>
__global__ __launch_bounds__(PARTS ? 1024 : 256) void rmsnorm_kernel(
    const std::conditional_t<PARTS, float, __hip_bfloat16>* __restrict__ x,
    const __hip_bfloat16* __restrict__ res,
    __hip_bfloat16* __restrict__ out,
    __hip_bfloat16* __restrict__ res_out,
    const __hip_bfloat16* __restrict__ weight,
    int H, float eps, int parts = 1, long step = 0) {
  const int row = blockIdx.x;
  const long base = (long)row * H;
  const int tid = threadIdx.x;
  const int nthr = blockDim.x;
  __shared__ float s_partial[16];

  shortx8 held[N > 0 ? N : 1], scale[N > 0 ? N : 1];
  if constexpr (N > 0)
#pragma unroll
    for (int k = 0; k < N; ++k)
      if ((tid + k * nthr) * 8 < H)
        scale[k] = *reinterpret_cast<const shortx8*>(weight + (tid + k * nthr) * 8);
  float ss = 0.f;
  // each thread strides over the row in 8-element vectors
  auto add = [&](int i, shortx8& kept) {
    float vals[8];
    if constexpr (PARTS) {
      add_parts8(vals, x + base + i, parts, step);
    } else {
      kept = *reinterpret_cast<const shortx8*>(x + base + i);
#pragma unroll
      for (int j = 0; j < 8; ++j) vals[j] = bf16_to_f32((unsigned short)kept[j]);
    }
    if (RESIDUAL) {
      shortx8 r = *reinterpret_cast<const shortx8*>(res + base + i);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        vals[j] += bf16_to_f32((unsigned short)r[j]);
        kept[j] = (short)f32_to_bf16(vals[j]);
      }
      *reinterpret_cast<shortx8*>(res_out + base + i) = kept;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) ss = fmaf(vals[j], vals[j], ss);  // (one order for every N)
  };
  if constexpr (N > 0) {
#pragma unroll
    for (int k = 0; k < N; ++k)
      if ((tid + k * nthr) * 8 < H) add((tid + k * nthr) * 8, held[k]);
  } else {
    for (int i = tid * 8; i < H; i += nthr * 8) add(i, held[0]);
  }
  ss = wave_sum(ss);
  const int wid = tid / WAVE, lid = tid % WAVE;
  if (lid == 0) s_partial[wid] = ss;
  __syncthreads();
  float all = 0.f;
  for (int w = 0; w < nthr / WAVE; ++w) all += s_partial[w];
  const float inv = rsqrtf(all / H + eps);
  auto write = [&](int i, const shortx8& v, const shortx8& w) {
    shortx8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      o[j] = (short)f32_to_bf16(bf16_to_f32((unsigned short)v[j]) * inv *
                                bf16_to_f32((unsigned short)w[j]));
    *reinterpret_cast<shortx8*>(out + base + i) = o;
  };
  if constexpr (N > 0) {
#pragma unroll
    for (int k = 0; k < N; ++k)
      if ((tid + k * nthr) * 8 < H) write((tid + k * nthr) * 8, held[k], scale[k]);
  } else {
    const __hip_bfloat16* src = RESIDUAL ? res_out : (const __hip_bfloat16*)x;
    for (int i = tid * 8; i < H; i += nthr * 8)
      write(i, *reinterpret_cast<const shortx8*>(src + base + i),
            *reinterpret_cast<const shortx8*>(weight + i));
  }
}

// Rows of up to 1024: a wave per row holds it in registers, so that it is read once and
// nothing goes through LDS (27700 rows of 768: 24 us for the norm alone with a workgroup
// per row, now 16 us; at 4096 a workgroup per row reads at 5.1 TB/s and stays).
template <bool RESIDUAL>
__global__ __launch_bounds__(256) void rmsnorm_wave_kernel(
    const __hip_bfloat16* __restrict__ x, const __hip_bfloat16* __restrict__ res,
    __hip_bfloat16* __restrict__ out, __hip_bfloat16* __restrict__ res_out,
    const __hip_bfloat16* __restrict__ weight, long T, int H, float eps) {
  const long row = blockIdx.x * 4L + threadIdx.x / WAVE;
  if (row >= T) return;
  const int lane = threadIdx.x % WAVE;
  const long base = row * H;
  shortx8 v[2];
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int i = (lane + k * WAVE) * 8;
    if (i >= H) continue;
    v[k] = *reinterpret_cast<const shortx8*>(x + base + i);
    shortx8 r;
    if (RESIDUAL) r = *reinterpret_cast<const shortx8*>(res + base + i);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float y = bf16_to_f32((unsigned short)v[k][j]);
      if (RESIDUAL) {
        y += bf16_to_f32((unsigned short)r[j]);
        v[k][j] = (short)f32_to_bf16(y);
      }
      ss += y * y;
    }
    if (RESIDUAL) *reinterpret_cast<shortx8*>(res_out + base + i) = v[k];
  }
  const float inv = rsqrtf(wave_sum(ss) / H + eps);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int i = (lane + k * WAVE) * 8;
    if (i >= H) continue;
    const shortx8 w = *reinterpret_cast<const shortx8*>(weight + i);
    shortx8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      o[j] = (short)f32_to_bf16(bf16_to_f32((unsigned short)v[k][j]) * inv *
                                bf16_to_f32((unsigned short)w[j]));
    *reinterpret_cast<shortx8*>(out + base + i) = o;
  }
}

template <bool RESIDUAL>
static void rmsnorm_launch(const torch::Tensor& x, const void* res, const torch::Tensor& out,
                           void* res_out, const torch::Tensor& weight, long T, int H,
                           double eps) {
  auto* xp = (const __hip_bfloat16*)x.data_ptr();
  auto* wp = (const __hip_bfloat16*)weight.data_ptr();
  auto* op = (__hip_bfloat16*)out.data_ptr();
  if (H <= 1024)
    hipLaunchKernelGGL(rmsnorm_wave_kernel<RESIDUAL>, dim3((T + 3) / 4), dim3(256), 0,
                       CUR_STREAM, xp, (const __hip_bfloat16*)res, op,
                       (__hip_bfloat16*)res_out, wp, T, H, (float)eps);
  else {
    auto launch = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(T), dim3(256), 0, CUR_STREAM, xp,
                         (const __hip_bfloat16*)res, op, (__hip_bfloat16*)res_out, wp, H,
                         (float)eps, 1, 0L);
    };
    if (H <= 2048) launch(rmsnorm_kernel<RESIDUAL, false, 1>);
    else if (H <= 4096) launch(rmsnorm_kernel<RESIDUAL, false, 2>);
    else if (H <= 8192) launch(rmsnorm_kernel<RESIDUAL, false, 4>);
    else launch(rmsnorm_kernel<RESIDUAL, false, 0>);
  }
  HIP_CHECK_KERNEL();
}

torch::Tensor rmsnorm(torch::Tensor x, torch::Tensor weight, double eps) {
  TORCH_CHECK(x.is_cuda() && x.dtype() == torch::kBFloat16, "rmsnorm: bf16 GPU only");
  TORCH_CHECK(x.size(-1) % 8 == 0, "H must be a multiple of 8");
  auto x2 = x.view({-1, x.size(-1)});
  auto out = torch::empty_like(x);
  int T = x2.size(0), H = x2.size(1);
  if (T == 0) return out;
  rmsnorm_launch<false>(x, nullptr, out, nullptr, weight, T, H, eps);
  return out;
}

std::vector<torch::Tensor> rmsnorm_residual(torch::Tensor x, torch::Tensor res,
                                            torch::Tensor weight, double eps) {
  // A product in parts: several, each of the residual's two dimensions. Nothing else is
  // float32: an activation has its residual's shape.
  if (x.dtype() == torch::kFloat32 && x.dim() == 3 && x.size(0) > 1) {
    const long S = x.size(0), T = x.size(1), H = x.size(2);
    TORCH_CHECK(x.is_cuda() && x.is_contiguous() && res.dtype() == torch::kBFloat16 &&
                    res.dim() == 2 && res.size(0) == T && res.size(1) == H && weight.numel() == H && H % 8 == 0,
                "parts [S, T, H] and residual [T, H]");
    const auto rc = res.contiguous();
    auto out = torch::empty_like(rc), res_out = torch::empty_like(rc);
    if (T == 0) return {out, res_out};
    const int threads = (int)std::min(1024L, (H / 8 + 63) / 64 * 64);
    const auto kern = H <= 8192 ? rmsnorm_kernel<true, true, 1> : rmsnorm_kernel<true, true, 0>;
    hipLaunchKernelGGL(kern, dim3(T), dim3(threads), 0, CUR_STREAM, x.data_ptr<float>(), (const __hip_bfloat16*)rc.data_ptr(),
                       (__hip_bfloat16*)out.data_ptr(), (__hip_bfloat16*)res_out.data_ptr(),
                       (const __hip_bfloat16*)weight.data_ptr(), (int)H, (float)eps, (int)S,
                       T * H);
    HIP_CHECK_KERNEL();
    return {out, res_out};
  }
  TORCH_CHECK(x.is_cuda() && x.dtype() == torch::kBFloat16, "bf16 GPU only");
  auto out = torch::empty_like(x);
  auto res_out = torch::empty_like(x);
  auto x2 = x.view({-1, x.size(-1)});
  int T = x2.size(0), H = x2.size(1);
  TORCH_CHECK(H % 8 == 0, "H must be a multiple of 8");
  if (T == 0) return {out, res_out};
  const auto rc = res.contiguous();
  rmsnorm_launch<true>(x, rc.data_ptr(), out, res_out.data_ptr(), weight, T, H, eps);
  return {out, res_out};
}

// --------------------------------------------------------------- silu_mul

__global__ void silu_mul_kernel(const __hip_bfloat16* __restrict__ gu,
                                __hip_bfloat16* __restrict__ out,
                                int T, int I) {
  // gu is [T, 2I]; out [T, I]; 8 elements per thread, grid-stride
  const long total = (long)T * I / 8;
  for (long idx = blockIdx.x * (long)blockDim.x + threadIdx.x; idx < total;
       idx += (long)gridDim.x * blockDim.x) {
    const long row = idx / (I / 8);
    const long col = (idx % (I / 8)) * 8;
    shortx8 g = *reinterpret_cast<const shortx8*>(gu + row * 2 * I + col);
    shortx8 u = *reinterpret_cast<const shortx8*>(gu + row * 2 * I + I + col);
    shortx8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float gf = bf16_to_f32((unsigned short)g[j]);
      float uf = bf16_to_f32((unsigned short)u[j]);
      float s = gf / (1.f + __expf(-gf));
      o[j] = (short)f32_to_bf16(s * uf);
    }
    *reinterpret_cast<shortx8*>(out + row * I + col) = o;
  }
}

torch::Tensor silu_mul(torch::Tensor gu) {
  TORCH_CHECK(gu.is_cuda() && gu.dtype() == torch::kBFloat16, "bf16 GPU only");
  int I2 = gu.size(-1);
  TORCH_CHECK(I2 % 16 == 0, "intermediate must be a multiple of 8");
  auto sizes = gu.sizes().vec();
  sizes.back() = I2 / 2;
  auto out = torch::empty(sizes, gu.options());
  auto gu2 = gu.view({-1, I2});
  int T = gu2.size(0), I = I2 / 2;
  if (T == 0) return out;
  long total = (long)T * I / 8;
  int blocks = (int)std::min<long>((total + 255) / 256, 2048);
  hipLaunchKernelGGL(silu_mul_kernel, dim3(blocks), dim3(256), 0,
                     CUR_STREAM,
                     (const __hip_bfloat16*)gu.data_ptr(),
                     (__hip_bfloat16*)out.data_ptr(), T, I);
  HIP_CHECK_KERNEL();
  return out;
}

// ------------------------------------------------------------------- rope

// In-place NeoX-pairing RoPE on q [T, Hq, D] and k [T, Hkv, D], whose rows may be strided.
// cos_sin: [max_pos, D] f32 (first half cos, second half sin).
// A thread per VEC pairs of a head (16-byte accesses at 8): bound by memory. 27700 rows of
// 24 heads of 64 took 104 us in 2-byte accesses (beside 54 us of copies of strided rows),
// now 32 us in place.
template <int VEC>
__global__ __launch_bounds__(256) void rope_kernel(
    __hip_bfloat16* __restrict__ q, __hip_bfloat16* __restrict__ k,
    const int* __restrict__ positions, const float* __restrict__ cos_sin, long T, int Hq,
    int Hkv, int D, long qstride, long kstride) {
  const int half = D / 2, parts = half / VEC, heads = Hq + Hkv;
  const long x = blockIdx.x * 256L + threadIdx.x;
  const long row = x / (heads * parts);
  if (row >= T) return;
  const int h = x % (heads * parts) / parts, i = x % parts * VEC;
  const float* cs = cos_sin + (long)positions[row] * D + i;
  unsigned short* base = (unsigned short*)(h < Hq ? q + row * qstride + (long)h * D
                                                  : k + row * kstride + (long)(h - Hq) * D) + i;
  unsigned short u[VEC], w[VEC];
  if constexpr (VEC == 8) {
    *(shortx8*)u = *(const shortx8*)base;
    *(shortx8*)w = *(const shortx8*)(base + half);
  } else {
    u[0] = base[0];
    w[0] = base[half];
  }
#pragma unroll
  for (int j = 0; j < VEC; ++j) {
    const float c = cs[j], s = cs[half + j], x1 = bf16_to_f32(u[j]), x2 = bf16_to_f32(w[j]);
    u[j] = f32_to_bf16(__builtin_fmaf(x1, c, -(x2 * s)));  // (packed attention has the same)
    w[j] = f32_to_bf16(__builtin_fmaf(x2, c, x1 * s));
  }
  if constexpr (VEC == 8) {
    *(shortx8*)base = *(const shortx8*)u;
    *(shortx8*)(base + half) = *(const shortx8*)w;
  } else {
    base[0] = u[0];
    base[half] = w[0];
  }
}

void rope_apply_(torch::Tensor q, torch::Tensor k, torch::Tensor positions,
                 torch::Tensor cos_sin) {
  TORCH_CHECK(q.is_cuda() && q.dtype() == torch::kBFloat16 && k.dtype() == q.dtype(),
              "bf16 GPU only");
  const long T = q.size(0);
  const int Hq = q.size(1), D = q.size(2), Hkv = k.size(1);
  for (auto* t : {&q, &k})  // (the stride of a single head says nothing)
    TORCH_CHECK(t->stride(2) == 1 && (t->stride(1) == D || t->size(1) == 1) &&
                    t->size(0) == T && t->size(2) == D,
                "heads of a row lie side by side");
  if (T == 0) return;
  auto cs = cos_sin.to(torch::kFloat32).contiguous();
  auto launch = [&](auto kern, int vec) {
    const long items = T * (Hq + Hkv) * (D / 2 / vec);
    hipLaunchKernelGGL(kern, dim3((items + 255) / 256), dim3(256), 0, CUR_STREAM,
                       (__hip_bfloat16*)q.data_ptr(), (__hip_bfloat16*)k.data_ptr(),
                       positions.data_ptr<int>(), cs.data_ptr<float>(), T, Hq, Hkv, D,
                       q.stride(0), k.stride(0));
  };
  const long odd = D / 2 | q.stride(0) | k.stride(0) | (long)q.data_ptr() >> 1 |
                   (long)k.data_ptr() >> 1;
  if (odd % 8 == 0) launch(rope_kernel<8>, 8);
  else launch(rope_kernel<1>, 1);
  HIP_CHECK_KERNEL();
}

// ---------------------------------------------------------- kv_cache_write

// Scatter new K/V rows into the paged cache.
// k/v: [T, Hkv, D]; caches: [NP, Hkv, P, D]; slot = page*P + off.
template <bool FP8>
__global__ void kv_cache_write_kernel(
    const __hip_bfloat16* __restrict__ k, const __hip_bfloat16* __restrict__ v,
    void* __restrict__ kc, void* __restrict__ vc,
    const int* __restrict__ slots, int T, int Hkv, int P, int D) {
  // one wave per (token, head); lane copies 8 elements at a time
  const int waves_per_block = blockDim.x / WAVE;
  const long wave_id = (long)blockIdx.x * waves_per_block + threadIdx.x / WAVE;
  const int lane = threadIdx.x % WAVE;
  if (wave_id >= (long)T * Hkv) return;
  const int t = wave_id / Hkv;
  const int h = wave_id % Hkv;
  const int slot = slots[t];
  if (slot < 0) return;
  const int page = slot / P, off = slot % P;
  const long src = ((long)t * Hkv + h) * D;
  const long dst = (((long)page * Hkv + h) * P + off) * D;
  for (int i = lane * 8; i < D; i += WAVE * 8) {
    if constexpr (FP8) {
      *reinterpret_cast<u64b*>((unsigned char*)kc + dst + i) =
          bf16x8_to_fp8x8(*reinterpret_cast<const shortx8*>(k + src + i));
      *reinterpret_cast<u64b*>((unsigned char*)vc + dst + i) =
          bf16x8_to_fp8x8(*reinterpret_cast<const shortx8*>(v + src + i));
    } else {
      *reinterpret_cast<shortx8*>((__hip_bfloat16*)kc + dst + i) =
          *reinterpret_cast<const shortx8*>(k + src + i);
      *reinterpret_cast<shortx8*>((__hip_bfloat16*)vc + dst + i) =
          *reinterpret_cast<const shortx8*>(v + src + i);
    }
  }
}

void kv_cache_write(torch::Tensor k, torch::Tensor v, torch::Tensor kc,
                    torch::Tensor vc, torch::Tensor slots) {
  TORCH_CHECK(k.is_cuda() && k.dtype() == torch::kBFloat16, "bf16 GPU only");
  int T = k.size(0), Hkv = k.size(1), D = k.size(2);
  int P = kc.size(2);
  if (T == 0) return;
  long waves = (long)T * Hkv;
  int wpb = 4;
  const bool fp8 = kc.dtype() == torch::kFloat8_e4m3fn;
  if (fp8)
    hipLaunchKernelGGL(kv_cache_write_kernel<true>,
                       dim3((waves + wpb - 1) / wpb), dim3(wpb * WAVE), 0,
                       CUR_STREAM, (const __hip_bfloat16*)k.data_ptr(),
                       (const __hip_bfloat16*)v.data_ptr(), kc.data_ptr(),
                       vc.data_ptr(), slots.data_ptr<int>(), T, Hkv, P, D);
  else
    hipLaunchKernelGGL(kv_cache_write_kernel<false>,
                       dim3((waves + wpb - 1) / wpb), dim3(wpb * WAVE), 0,
                       CUR_STREAM, (const __hip_bfloat16*)k.data_ptr(),
                       (const __hip_bfloat16*)v.data_ptr(), kc.data_ptr(),
                       vc.data_ptr(), slots.data_ptr<int>(), T, Hkv, P, D);
  HIP_CHECK_KERNEL();
}

// ------------------------------------------------- fused qkv post-process
// One kernel replaces: q/k/v slice copies (the qkv GEMM output is sliced
// non-contiguously), RoPE on q and k, and the paged-cache K/V scatter —
// rocprof showed those as ~5 launches + 3 copies per layer of pure launch
// floor in the decode step.
// qkv: [T, (Hq+2*Hkv)*D] -> writes q_out [T, Hq, D] (roped), kc/vc slots.
// PARTS: qkv is a product in `parts` fp32 terms `step` apart, see rmsnorm_kernel. Beside a
// whole product that costs 0.3 us for 96 rows of 6144 in 2 parts and 0.4 for 23 of 3072 in 5
// (warm cache pages). Slot and position are asked for before anything else, so that few
// rows make two trips to memory and not three: of cold cache pages 23 of 3072 in 5 parts 3.82 us
// and 3.66, 96 of 6144 in 2 parts 4.46 and 4.18.
// bias: one term more per column or null, added to the rounded product.
// A thread per VEC columns of a head and their partners half a head on (16-byte accesses
// at 8): bound by memory. 6172 rows of 48 heads of 128 took 58 us in 2-byte accesses,
// now 26; 3000 rows of 48 heads of 64 27 and 8.5.
template <bool FP8, bool PARTS, int VEC>
__global__ __launch_bounds__(256) void fused_rope_kv_write_kernel(
    const std::conditional_t<PARTS, float, unsigned short>* __restrict__ qkv,
    const unsigned short* __restrict__ bias,
    __hip_bfloat16* __restrict__ q_out,
    void* __restrict__ kc, void* __restrict__ vc,
    const int* __restrict__ positions, const int* __restrict__ slots,
    const float* __restrict__ cos_sin,
    int T, int Hq, int Hkv, int D, int P, int parts, long step) {
  const int half = D / 2, HT = Hq + 2 * Hkv;
  const unsigned units = half / VEC, x = blockIdx.x * 256u + threadIdx.x;
  const unsigned unit_row = x / units;
  if (unit_row >= (unsigned)T * HT) return;
  const int i = (x - unit_row * units) * VEC, t = unit_row / HT, h = unit_row - t * HT;
  const long row = unit_row;
  const bool is_q = h < Hq, is_v = h >= Hq + Hkv;
  // (asked for before anything that is read waits for them)
  const int slot = is_q ? 0 : slots[t], position = is_v ? 0 : positions[t];
  float y[2][VEC];  // columns i.. and half + i..
#pragma unroll
  for (int z = 0; z < 2; ++z) {
    const auto* src = qkv + row * D + z * half + i;
    if constexpr (PARTS && VEC == 8) {
      add_parts8(y[z], src, parts, step);
    } else if constexpr (PARTS) {
      float sum = 0.f;
#pragma unroll 4
      for (int p = 0; p < parts; ++p) sum += src[p * step];
      y[z][0] = bf16_to_f32(f32_to_bf16(sum));
    } else if constexpr (VEC == 8) {
      const shortx8 v = *reinterpret_cast<const shortx8*>(src);
#pragma unroll
      for (int j = 0; j < 8; ++j) y[z][j] = bf16_to_f32((unsigned short)v[j]);
    } else {
      y[z][0] = bf16_to_f32(src[0]);
    }
    if (bias) {
      const unsigned short* b = bias + (long)h * D + z * half + i;
#pragma unroll
      for (int j = 0; j < VEC; ++j)
        y[z][j] = bf16_to_f32(f32_to_bf16(y[z][j] + bf16_to_f32(b[j])));
    }
  }
  if (slot < 0) return;
  long dst = ((long)t * Hq + h) * D + i;
  if (!is_q) {
    const int head = h - Hq - (is_v ? Hkv : 0);
    dst = (((long)(slot / P) * Hkv + head) * P + slot % P) * D + i;
  }
  if (!is_v) {
    const float* cs = cos_sin + (long)position * D + i;
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const float c = cs[j], s = cs[half + j], x1 = y[0][j], x2 = y[1][j];
      // (the compiler's own choices for the two forms, held fast: decode attention that rotates
      // by itself has either's bits)
      y[0][j] = __builtin_fmaf(x1, c, -(x2 * s));
      y[1][j] = VEC == 8 ? __builtin_fmaf(x1, s, x2 * c) : __builtin_fmaf(x2, c, x1 * s);
    }
  }
  void* to = is_q ? (void*)q_out : is_v ? vc : kc;
#pragma unroll
  for (int z = 0; z < 2; ++z) {
    const long at = dst + z * half;
    if (FP8 && !is_q) {
      unsigned char out[VEC];
#pragma unroll
      for (int j = 0; j < VEC; ++j) out[j] = f32_to_fp8(y[z][j]);
      if constexpr (VEC == 8) *reinterpret_cast<u64b*>((unsigned char*)to + at) = *(u64b*)out;
      else ((unsigned char*)to)[at] = out[0];
    } else {
      unsigned short out[VEC];
#pragma unroll
      for (int j = 0; j < VEC; ++j) out[j] = f32_to_bf16(y[z][j]);
      if constexpr (VEC == 8)
        *reinterpret_cast<shortx8*>((unsigned short*)to + at) = *(shortx8*)out;
      else ((unsigned short*)to)[at] = out[0];
    }
  }
}

bool rotates_by_eight(long T, long width) { return T * width >= 1 << 20; }

torch::Tensor fused_rope_kv_write(torch::Tensor qkv, torch::Tensor positions,
                                  torch::Tensor slots, torch::Tensor cos_sin,
                                  torch::Tensor kc, torch::Tensor vc,
                                  long Hq, long Hkv, c10::optional<torch::Tensor> bias) {
  const bool raw = qkv.dtype() == torch::kFloat32 && qkv.dim() == 3;  // a product in parts
  TORCH_CHECK(qkv.is_cuda() && (raw ? qkv.is_contiguous() : qkv.dtype() == torch::kBFloat16),
              "bf16 GPU only");
  const int T = qkv.size(raw ? 1 : 0);
  const int P = kc.size(2), D = kc.size(3);
  const long width = (Hq + 2 * Hkv) * D;
  TORCH_CHECK(qkv.size(-1) == width, "qkv width mismatch");
  TORCH_CHECK(!bias || (bias->is_cuda() && bias->dtype() == torch::kBFloat16 &&
                        bias->is_contiguous() && bias->numel() == width),
              "a contiguous bf16 bias per column");
  auto q_out = torch::empty({(long)T, Hq, (long)D}, qkv.options().dtype(torch::kBFloat16));
  if (T == 0) return q_out;
  TORCH_CHECK(D % 2 == 0, "head width");
  uintptr_t bits = 0;
  for (const void* p : {(const void*)qkv.data_ptr(), (const void*)q_out.data_ptr(),
                        (const void*)kc.data_ptr(), (const void*)vc.data_ptr()})
    bits |= (uintptr_t)p;
  // few rows leave the chip idle with eight columns a thread: 23 rows of 3072 in 5 parts
  // 3.5 us and 2.8, but 300 rows of 4608 6.2 us both ways
  const int vec = D % 16 == 0 && bits % 16 == 0 && rotates_by_eight(T, width) ? 8 : 1;
  const long threads = (long)T * (Hq + 2 * Hkv) * (D / 2 / vec);
  TORCH_CHECK(threads < 1L << 32, "more rows than a launch can index");
  auto launch = [&](auto kern, auto* src) {
    hipLaunchKernelGGL(kern, dim3((threads + 255) / 256), dim3(256), 0, CUR_STREAM,
                       src, bias ? (const unsigned short*)bias->data_ptr() : nullptr,
                       (__hip_bfloat16*)q_out.data_ptr(), kc.data_ptr(), vc.data_ptr(),
                       positions.data_ptr<int>(), slots.data_ptr<int>(),
                       cos_sin.data_ptr<float>(), T, (int)Hq, (int)Hkv, D, P,
                       raw ? (int)qkv.size(0) : 1, T * width);
  };
  const auto* f = (const float*)qkv.data_ptr();
  const auto* h = (const unsigned short*)qkv.data_ptr();
#define ROPE(F8, VEC)                                               \
  if (raw) launch(fused_rope_kv_write_kernel<F8, true, VEC>, f);    \
  else launch(fused_rope_kv_write_kernel<F8, false, VEC>, h)
  if (kc.dtype() == torch::kFloat8_e4m3fn) {
    if (vec == 8) { ROPE(true, 8); } else { ROPE(true, 1); }
  } else {
    if (vec == 8) { ROPE(false, 8); } else { ROPE(false, 1); }
  }
#undef ROPE
  HIP_CHECK_KERNEL();
  return q_out;
}
