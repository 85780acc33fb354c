// Routed experts with a clamped GLU,
//     act = g sigmoid(alpha g) (u + shift),  g = min(gate, limit), u = clamp(up)
// (without a limit, alpha 1 and shift 0: silu(gate) up), or a squared relu, act =
// max(up, 0)^2, chosen by one of three routers:
//     z = W_r h + b (fp32; without b rounded to the weights' type, as such models' plain
//     product leaves it), the ``top`` largest, softmax over the chosen;
//     s = sigmoid(W_r h) (fp32), the ``top`` largest of s + c among the best groups of
//     neighbours (by the sum of their two largest), weights s / sum s * scale;
//     s = softmax(W_r h) (fp32) over all, the ``top`` largest among the best groups (by
//     their largest), weights s * scale
// as route -> sort -> gathered up product with the activation in its epilogue
// -> down product. Rows stay sorted by expert; the residual-norm kernel adds
// each token's weighted rows, so no scatter pass exists. Nothing is read back
// to the host and all shapes are static: prompts and captured decode steps run
// the same code, only the row tile differs. A grid block looks up its (expert,
// row tile) in a device table; blocks past its end leave at once, so experts
// nobody chose cost no weight traffic.
#include "elem.h"
#include "flash_tiles.h"
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

#define CUR_STREAM c10::hip::getCurrentHIPStream().stream()
#define MAX_EXPERTS 1024

union mfrag {
  shortx8 s;
  bf16x8 v;
};

// ------------------------------------------------------------------- router

enum { CHOSEN_SOFTMAX = 0, GROUPED_SIGMOID = 1, GROUPED_SOFTMAX = 2 };

// The largest value of a wave's lanes but NaN, without a trip through LDS. (Choices by
// butterflies over value and index took 12 such trips each: 64 tokens of 2048 over 64
// experts, six each, 16.9 and 14.4 us; over 128, eight each, 28.7 and 25.8; 32 of 4096 over 8,
// two each, 10.5 and 9.6. What was left is a CU's read of the whole router.)
DEVINL float lanes_max(float x) {
  auto step = [](float a, auto CTRL) {
    return fmaxf(a, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(
        __builtin_bit_cast(int, a), decltype(CTRL)::value, 0xf, 0xf, false)));
  };
  x = step(x, std::integral_constant<int, 0xb1>{});   // neighbours
  x = step(x, std::integral_constant<int, 0x4e>{});   // pairs of a quad
  x = step(x, std::integral_constant<int, 0x141>{});  // halves of eight
  x = step(x, std::integral_constant<int, 0x140>{});  // of sixteen
  const unsigned u = __builtin_bit_cast(unsigned, x);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  x = fmaxf(__builtin_bit_cast(float, (unsigned)a[0]), __builtin_bit_cast(float, (unsigned)a[1]));
  const unsigned w = __builtin_bit_cast(unsigned, x);
  const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  return fmaxf(__builtin_bit_cast(float, (unsigned)b[0]), __builtin_bit_cast(float, (unsigned)b[1]));
}

// A wave chooses token t's experts. z: its logits, which are used up; score: 512 + groups
// floats for plain scores and the groups'.
template <int ROUTER>
DEVINL void choose(float* z, float* score, int lane, const float* bias, int* sel, float* gate,
                   int t, int E, int top, int groups, int keep, float scale) {
  constexpr bool GROUPED = ROUTER != CHOSEN_SOFTMAX;
  if constexpr (GROUPED) {
    float* gs = score + 512;
    const int n = E / groups;
    auto sync = [] {
      __threadfence_block();
      __builtin_amdgcn_wave_barrier();
    };
    if constexpr (ROUTER == GROUPED_SIGMOID) {
      for (int e = lane; e < E; e += WAVE) {
        score[e] = sigmoid_f(z[e]);
        z[e] = score[e] + bias[e];
      }
    } else {
      float most = -INFINITY, all = 0.f;
      for (int e = lane; e < E; e += WAVE) most = fmaxf(most, z[e]);
      most = wave_max(most);
      for (int e = lane; e < E; e += WAVE) all += score[e] = expf(z[e] - most);
      all = wave_sum(all);
      for (int e = lane; e < E; e += WAVE) score[e] /= all;
    }
    sync();
    for (int x = lane; x < groups; x += WAVE) {
      float a = -INFINITY, b = -INFINITY;  // the two largest
      for (int e = x * n; e < (x + 1) * n; ++e) {
        const float c = z[e];
        b = fmaxf(b, fminf(a, c));
        a = fmaxf(a, c);
      }
      gs[x] = ROUTER == GROUPED_SIGMOID && n > 1 ? a + b : a;
    }
    sync();
    for (int x = lane; x < groups; x += WAVE) {
      int better = 0;
      for (int o = 0; o < groups; ++o)
        better += gs[o] > gs[x] || (gs[o] == gs[x] && o < x);
      if (better >= keep)
        for (int e = x * n; e < (x + 1) * n; ++e) z[e] = -INFINITY;
    }
    sync();
  }
  float first = 0.f, sum = 0.f;
  // up to 64 experts: a lane holds its own, the first of the largest is found by lane
  const bool few = E <= WAVE;
  float mine = few && lane < E ? z[lane] : -INFINITY;
  // up to 64 choices: a lane holds one (stored one by one, each waited for the one before)
  const bool hold = top <= WAVE;
  int my_at = 0;
  float my_p = 0.f;
  for (int n = 0; n < top; ++n) {
    float best = -INFINITY;
    int at = 0x7fffffff;
    if (few) {
      best = lanes_max(mine);
      const unsigned long long who = __ballot(mine == best && best > -INFINITY);
      if (who) at = __builtin_ctzll(who);
      else best = -INFINITY;
      if (lane == at) mine = -INFINITY;
    } else {
      float own = -INFINITY;
      int oat = 0;
      for (int e = lane; e < E; e += WAVE)
        if (z[e] > own) { own = z[e]; oat = e; }
      best = lanes_max(own);
      for (unsigned long long who = __ballot(own == best && best > -INFINITY); who;
           who &= who - 1)
        at = min(at, __builtin_amdgcn_readlane(oat, __builtin_ctzll(who)));
    }
    at = min(at, E - 1);  // all logits NaN: still a valid expert
    if (n == 0) first = best;
    const float p = GROUPED ? score[at] : expf(best - first);
    sum += p;
    if (lane == n % WAVE) {
      my_at = at;
      my_p = p;
      if (!hold) {
        sel[(long)t * top + n] = at;
        gate[(long)t * top + n] = p;
      }
    }
    if (few) continue;
    if (lane == 0) z[at] = -INFINITY;
    __threadfence_block();
    __builtin_amdgcn_wave_barrier();
  }
  auto scaled = [&](float w) {
    return ROUTER == GROUPED_SIGMOID ? w / (sum + 1e-20f) * scale
           : ROUTER == GROUPED_SOFTMAX ? w * scale : w / sum;
  };
  if (hold) {
    if (lane < top) {
      sel[(long)t * top + lane] = my_at;
      gate[(long)t * top + lane] = scaled(my_p);
    }
    return;
  }
  // each lane rescales what it wrote
  for (int n = lane; n < top; n += WAVE) {
    float& w = gate[(long)t * top + n];
    w = scaled(w);
  }
}

// a logit as it is chosen by: without a bias those of a product in the model's own type
template <typename T, int ROUTER>
DEVINL float whole_logit(float z, const float* bias, int e) {
  if (ROUTER != CHOSEN_SOFTMAX) return z;
  return bias ? z + bias[e] : sizeof(T) == 2 ? bf16_to_f32(f32_to_bf16(z)) : z;
}

// The choices alone, of logits in S parts [S, T, E] to be added: a wave per token.
template <int ROUTER>
__global__ __launch_bounds__(WAVE) void moe_choose_kernel(
    const float* __restrict__ part, int S, const float* __restrict__ bias,
    int* __restrict__ sel, float* __restrict__ gate, int E, int top, int groups, int keep,
    float scale) {
  extern __shared__ float score[];  // [512 + 512], then logits
  float* z = score + 1024;
  const int t = blockIdx.x, lane = threadIdx.x;
  const long step = (long)gridDim.x * E;
  for (int e = lane; e < E; e += WAVE) {
    const float* p = part + (long)t * E + e;
    float sum = 0.f;
    for (int s = 0; s < S; s += 8) {  // asked for together
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = p[min(s + u, S - 1) * step];
#pragma unroll
      for (int u = 0; u < 8; ++u) sum += s + u < S ? v[u] : 0.f;
    }
    z[e] = whole_logit<bf16_t, ROUTER>(sum, bias, e);
  }
  __threadfence_block();
  __builtin_amdgcn_wave_barrier();
  choose<ROUTER>(z, score, lane, bias, sel, gate, t, E, top, groups, keep, scale);
}

// One workgroup per 16 tokens; its waves split the contraction. GROUPED_SIGMOID: bias
// is the scores' correction; GROUPED_SOFTMAX: there is none.
template <typename T, bool MATRIX16, int ROUTER>
__global__ __launch_bounds__(1024) void moe_route_kernel(
    const T* __restrict__ h, const T* __restrict__ router,
    const float* __restrict__ bias, int* __restrict__ sel, float* __restrict__ gate,
    int T_, int W, int E, int top, int groups, int keep, float scale) {
  extern __shared__ float logits[];  // [16][E]
  __shared__ float part[16][16][64];
  const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
  const int i = lane & 15, g = lane >> 4;
  const int t0 = blockIdx.x * 16;
  const long arow = (long)min(t0 + i, T_ - 1) * W;
  for (int e0 = 0; e0 < E; e0 += 64) {
    floatx4 acc[4];
    long brow[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
      brow[j] = (long)min(e0 + j * 16 + i, E - 1) * W;
    }
    if constexpr (MATRIX16) {  // bf16 operands, W a multiple of 8
      for (int k = wave * 32; k < W; k += 512) {
        const int kk = k + g * 8;
        mfrag a, b;
        a.s = shortx8{0, 0, 0, 0, 0, 0, 0, 0};
        b.s = a.s;
        if (kk < W) a.s = *reinterpret_cast<const shortx8*>(h + arow + kk);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (e0 + j * 16 >= E) break;
          if (kk < W) b.s = *reinterpret_cast<const shortx8*>(router + brow[j] + kk);
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, acc[j], 0, 0, 0);
        }
      }
    } else {
      for (int k = wave * 4; k < W; k += 64) {
        const int kk = k + g;
        const float a = kk < W ? ldf(h + arow + kk) : 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (e0 + j * 16 >= E) break;
          const float b = kk < W ? ldf(router + brow[j] + kk) : 0.f;
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc[j], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) part[wave][4 * g + r][j * 16 + i] = acc[j][r];
    __syncthreads();
    {
      const int t = threadIdx.x / 64, x = threadIdx.x % 64, e = e0 + x;
      float z = 0.f;
#pragma unroll
      for (int v = 0; v < 16; ++v) z += part[v][t][x];
      if (e < E) logits[t * E + e] = whole_logit<T, ROUTER>(z, bias, e);
    }
    __syncthreads();
  }
  if (t0 + wave < T_)
    choose<ROUTER>(logits + wave * E, &part[wave][0][0], lane, bias, sel, gate, t0 + wave, E,
                   top, groups, keep, scale);
}

torch::Tensor router_rows(const torch::Tensor& x, const torch::Tensor& w);  // of few_rows.hip

// Few tokens: a workgroup for 16 of them reads the whole router, at some 25 GB/s of a CU, where
// the products' kernel of few rows spreads it and the tokens over 8 and more, and a second launch
// adds the parts and chooses. Both give the same bits. Cold routers, us, whole and in parts, of 1,
// 4, 8, 16, 64 and 128 tokens:
//   E x W       1              4             8             16            64            128
//   8 x 4096    6.4 and 6.5    7.4 and 6.9   8.1 and 6.8   10.2 and 7.0  10.3 and 7.1  10.3 and 7.1
//   16 x 2880   6.5 and 6.3    7.2 and 6.6   7.8 and 6.5   9.3 and 6.6   9.5 and 6.8   9.5 and 6.9
//   64 x 2048   10.9 and 5.8   11.4 and 6.4  12.0 and 6.4  13.3 and 6.4  13.5 and 6.5  13.6 and 6.5
//   128 x 4096  34.6 and 8.9   36.2 and 9.6  37.5 and 9.8  40.7 and 9.8  41.2 and 9.9  41.3 and 10.4
//   8 x 2880    5.6 and 6.5    6.4 and 6.6   6.8 and 6.7   8.4 and 6.9   8.7 and 6.9   8.7 and 7.0
//   16 x 2048   5.6 and 5.8    6.1 and 6.1   6.6 and 6.3   8.0 and 6.3   8.2 and 6.5   8.1 and 6.5
//   32 x 1024   5.3 and 5.9    5.9 and 6.0   6.2 and 6.0   7.1 and 6.2   7.3 and 6.3   7.3 and 6.3
//   64 x 512    5.2 and 5.7    5.6 and 5.9   5.9 and 6.0   6.7 and 6.1   6.9 and 6.2   6.9 and 6.2
//   12 x 1536   4.8 and 6.1    5.4 and 6.3   5.7 and 6.3   6.9 and 6.3   7.1 and 6.5   7.1 and 6.5
//   16 x 1024   4.6 and 5.6    4.9 and 5.9   5.3 and 6.0   6.2 and 6.1   6.5 and 6.2   6.4 and 6.3
//   8 x 1024    4.2 and 5.9    4.6 and 6.2   5.0 and 6.3   5.9 and 6.3   6.2 and 6.4   6.2 and 6.4
// The line is what the first workgroup reads, 40000 values: at it (16 x 2048, 4 tokens; 32 x 1024,
// 8; 64 x 512, 16) the two are alike or parts ahead; what it gives up is 0.4 us of 128 x 256.
static bool route_in_parts(const torch::Tensor& h, const torch::Tensor& router) {
  const long T_ = h.size(0), W = h.size(1), E = router.size(0);
  return h.dtype() == torch::kBFloat16 && T_ <= 128 && W % 64 == 0 && W >= 256 &&
         W * (E + std::min(T_, 16L)) >= 40000 && (uintptr_t)router.data_ptr() % 16 == 0 &&
         (uintptr_t)h.data_ptr() % 16 == 0;
}

template <int ROUTER>
static std::vector<torch::Tensor> route(const torch::Tensor& h, const torch::Tensor& router,
                                        const c10::optional<torch::Tensor>& bias, long top,
                                        long groups, long keep, double scale) {
  TORCH_CHECK(h.is_cuda() && h.dim() == 2 && h.is_contiguous() &&
              router.is_contiguous() && router.dtype() == h.dtype());
  const long T_ = h.size(0), W = h.size(1), E = router.size(0);
  TORCH_CHECK(router.size(1) == W);
  TORCH_CHECK(bias ? ROUTER != GROUPED_SOFTMAX && bias->numel() == E &&
                         bias->dtype() == torch::kFloat32
                   : ROUTER != GROUPED_SIGMOID, "router bias");
  TORCH_CHECK(top >= 1 && top <= E && E <= 512, "1 <= top <= experts <= 512");
  auto sel = torch::empty({T_, top}, h.options().dtype(torch::kInt32));
  auto gate = torch::empty({T_, top}, h.options().dtype(torch::kFloat32));
  if (T_ == 0) return {sel, gate};
  if (route_in_parts(h, router)) {
    const auto part = router_rows(h, router);
    hipLaunchKernelGGL(moe_choose_kernel<ROUTER>, dim3(T_), dim3(WAVE), (1024 + E) * 4, CUR_STREAM,
                       part.template data_ptr<float>(), (int)part.size(0),
                       bias ? bias->data_ptr<float>() : nullptr, sel.data_ptr<int>(),
                       gate.data_ptr<float>(), (int)E, (int)top, (int)groups, (int)keep,
                       (float)scale);
    HIP_CHECK_KERNEL();
    return {sel, gate};
  }
  DISPATCH_ELEM(h.dtype() == torch::kBFloat16, {
    auto launch = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3((T_ + 15) / 16), dim3(1024), 16 * E * 4, CUR_STREAM,
                         (const T*)h.data_ptr(), (const T*)router.data_ptr(),
                         bias ? bias->data_ptr<float>() : nullptr, sel.data_ptr<int>(),
                         gate.data_ptr<float>(), (int)T_, (int)W, (int)E, (int)top,
                         (int)groups, (int)keep, (float)scale);
    };
    constexpr bool B16 = sizeof(T) == 2;
    if (B16 && W % 8 == 0) launch(moe_route_kernel<T, B16, ROUTER>);
    else launch(moe_route_kernel<T, false, ROUTER>);
  });
  HIP_CHECK_KERNEL();
  return {sel, gate};
}

std::vector<torch::Tensor> moe_route(torch::Tensor h, torch::Tensor router,
                                     c10::optional<torch::Tensor> bias, long top) {
  return route<CHOSEN_SOFTMAX>(h, router, bias, top, 1, 1, 1.0);
}

// sigmoid scores with a correction, softmax scores without
std::vector<torch::Tensor> moe_route_grouped(torch::Tensor h, torch::Tensor router,
                                             c10::optional<torch::Tensor> correction,
                                             long top, long groups, long keep, double scale) {
  const long E = router.size(0);
  TORCH_CHECK(groups >= 1 && E % groups == 0 && keep >= 1 && keep <= groups &&
              top <= keep * (E / groups), "expert groups");
  if (!correction) return route<GROUPED_SOFTMAX>(h, router, correction, top, groups, keep, scale);
  return route<GROUPED_SIGMOID>(h, router, correction, top, groups, keep, scale);
}

// --------------------------------------------------------------------- sort

// Rounds of the 256-row tile's workgroups, one a CU: as long as their tiles are high, 32 rows
// a step, and a constant; one that does not fill the chip leaves the others a higher clock.
// (4096 x 28672 x 4096: rounds of 256, 224, 192 and 128 rows 94, 84, 73 and 53 us; 1000 x 4096
// x 4096, 64 tiles of 256 rows 70 us, 128 of 128 41.)
__host__ __device__ inline float rounds_time(long tiles, float mean, int most) {
  const long full = tiles / 256, rest = tiles % 256;
  return full * (mean + 1.25f) + (rest ? (0.75f + 0.25f / 256 * rest) * (most + 1.25f) : 0.f);
}

// place[a]: sorted row of choice a; token[row]: its token; tables of the row tiles of the up
// and of the down product: (expert, first row, rows) of every tile, then expert -1; behind
// ``tiles`` of them their number. Tiles of TM rows; where that is 256 (and the tables are
// two) of at most 256, 32 at a time, an expert's all alike, and so many that the products'
// rounds, of ``cols`` tiles a row tile, are short (8 experts of 4096 x 14336, two each, 300
// tokens 711 and 575 us, 1000 tokens 821 to 816: where rows are many, tiles were many before).
// (The heights were weighed by a lane each, over all experts in turn: 512 of 1024 x 512, eight
// each, 3300 tokens 435 and 357 us for the whole; 64 of 2048 x 1408, six each, 400 tokens 248 and
// 239.)
__global__ __launch_bounds__(1024) void moe_sort_kernel(
    const int* __restrict__ sel, int A, int E, int top, int TM, int tiles, int cols_up,
    int cols_dn, int* __restrict__ place, int* __restrict__ token, int* __restrict__ table) {
  __shared__ int count[MAX_EXPERTS], base[MAX_EXPERTS], tbase[MAX_EXPERTS];
  __shared__ int s_high[2];
  const int tid = threadIdx.x;
  const bool even = TM == 256;
  for (int e = tid; e < E; e += 1024) count[e] = 0;
  __syncthreads();
  for (int a = tid; a < A; a += 1024) atomicAdd(&count[sel[a]], 1);
  __syncthreads();
  if (even && tid < WAVE) {  // tiles, and the highest of them, at each of five heights
    int parts = 0, nt[5] = {}, most[5] = {};
    for (int e = tid; e < E; e += WAVE) {
      const int u = (count[e] + 31) / 32;
      parts += u;
#pragma unroll
      for (int x = 0; x < 5; ++x) {
        const int n = (u + 3 + x) / (4 + x);
        nt[x] += n;
        most[x] = max(most[x], (u + n - 1) / max(n, 1));
      }
    }
#pragma unroll
    for (int off = 1; off < WAVE; off <<= 1) {
      parts += __shfl_xor(parts, off, WAVE);
#pragma unroll
      for (int x = 0; x < 5; ++x) {
        nt[x] += __shfl_xor(nt[x], off, WAVE);
        most[x] = max(most[x], __shfl_xor(most[x], off, WAVE));
      }
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      float low = 0.f;
      int best = 8;
#pragma unroll
      for (int x = 4; x >= 0; --x) {
        const float t = rounds_time((long)nt[x] * (k ? cols_dn : cols_up),
                                    (float)parts / max(nt[x], 1), most[x]);
        if (x == 4 || t < low) low = t, best = 4 + x;
      }
      if (tid == 0) s_high[k] = best;
    }
  }
  __syncthreads();
  for (int k = 0; k < (even ? 2 : 1); ++k, table += (tiles + 1) * 3) {
    const int step = even ? s_high[k] * 32 : TM;
    if (tid < WAVE) {  // exclusive sums over experts, one wave
      int rows = 0, nt = 0;
      for (int e0 = 0; e0 < E; e0 += WAVE) {
        const int e = e0 + tid;
        const int c = e < E ? count[e] : 0, n = (c + step - 1) / step;
        int sc = c, sk = n;
#pragma unroll
        for (int off = 1; off < WAVE; off <<= 1) {
          const int a = __shfl_up(sc, off, WAVE), b = __shfl_up(sk, off, WAVE);
          if (tid >= off) { sc += a; sk += b; }
        }
        if (e < E) { base[e] = rows + sc - c; tbase[e] = nt + sk - n; }
        rows += __shfl(sc, WAVE - 1, WAVE);
        nt += __shfl(sk, WAVE - 1, WAVE);
      }
      for (int t = nt + tid; t < tiles; t += WAVE) table[t * 3] = -1;
      if (tid == 0) table[tiles * 3] = nt;
    }
    __syncthreads();
    for (int e = tid; e < E; e += 1024) {
      const int c = count[e], n = (c + step - 1) / step, parts = (c + 31) / 32;
      for (int x = 0; x < n; ++x) {
        const int r = even ? x * parts / n * 32 : x * TM;
        const int end = even ? (x + 1) * parts / n * 32 : r + TM;
        int* t = table + (tbase[e] + x) * 3;
        t[0] = e;
        t[1] = base[e] + r;
        t[2] = min(end, c) - r;
      }
    }
    __syncthreads();
  }
  for (int a = tid; a < A; a += 1024) {
    const int row = atomicAdd(&base[sel[a]], 1);
    place[a] = row;
    token[row] = a / top;
  }
}

// ------------------------------------------------------------ grouped product

// what the product's epilogue does
enum { NO_ACT = 0, GLU_ACT = 1, RELU2_ACT = 2, SILU_ACT = 3 };

struct GroupArgs {
  const void* x;       // rows [*, K]; row r of the sorted batch is x[gather[r]]
  const int* gather;   // null: x itself is sorted
  const void* w;       // [E, N, K]; GLU: [E, 2N, K], gate rows then up rows
  void* y;             // [A, N]
  const int* table;    // of moe_sort_kernel; null: one expert for all ``rows``
  int N, K;
  float limit, alpha, shift;
  int rows = 0;        // of x
  bool silu = false;   // no limit, alpha 1 and shift 0, with silu_mul's exponential
  int ldx = 0;         // from row to row of x where that is not K (256-row tile only)
};

// x / d for d >= 1, once corrected: what replaces a division in the 256-row tile, whose
// results are bf16 and which has nothing to hide it behind. silu is as near to 64 bits with it
// as with a division (off by 1.75e-7 of itself at most, 3.7e-8 rms, -85 to 20), and 4 prompts
// of 2000 tokens, 8 experts of 4096 x 14336, lose half of the 2% that a division costs. (2^(x
// log2 e) in place of expf saves another 1% and is off by 3.9e-6; with the product's rounding
// brought in by 2.3e-7.) 0 where d is 2^126 or more.
DEVINL float over(float x, float d) {
  const float r = __builtin_amdgcn_rcpf(d), q = x * r;
  return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-d, q, x), r, q), d, x);
}

template <bool TILE256 = false>
DEVINL float clamped_glu(float g, float u, const GroupArgs& p) {
  // (fminf and fmaxf would drop a NaN)
  g = __builtin_elementwise_minimum(g, p.limit);
  u = __builtin_elementwise_minimum(__builtin_elementwise_maximum(u, -p.limit), p.limit);
  const float d = 1.f + expf(-p.alpha * g);
  // the gate first: a closed one makes nothing of however large an ``up``
  return (TILE256 ? over(g, d) : g / d) * (u + p.shift);
}

// silu(g) u with the exponential of silu_mul and the products of few rows
DEVINL float silu_glu(float g, float u) {
  return over(g, 1.f + __builtin_amdgcn_exp2f(-LOG2E * g)) * u;
}

// Any size and float32: 32 rows x 64 columns, 16 of K at a time, through LDS as
// fp32 (GLU: 32 gate and the matching 32 up columns).
template <typename T, int ACT>
__global__ __launch_bounds__(256) void grouped_any_kernel(GroupArgs p) {
  constexpr bool GLU = ACT == GLU_ACT;
  const int* tb = p.table + blockIdx.y * 3;
  const int e = tb[0];
  if (e < 0) return;
  const int row0 = tb[1], cnt = tb[2];
  __shared__ float xs[32][17], ws[64][17], cs[32][65];
  const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
  const int i = lane & 15, g = lane >> 4;
  constexpr int BN = GLU ? 32 : 64;
  const int n0 = blockIdx.x * BN;
  const T* w = (const T*)p.w + (long)e * (GLU ? 2 : 1) * p.N * p.K;
  floatx4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  for (int k0 = 0; k0 < p.K; k0 += 16) {
    __syncthreads();
    for (int x = tid; x < 32 * 16; x += 256) {
      const int r = x / 16, k = k0 + x % 16;
      const long src = row0 + min(r, cnt - 1);
      xs[r][x % 16] = k < p.K ? ldf((const T*)p.x + (long)(p.gather ? p.gather[src] : src) *
                                    p.K + k) : 0.f;
    }
    for (int x = tid; x < 64 * 16; x += 256) {
      const int r = x / 16, k = k0 + x % 16;
      const int c = n0 + (GLU ? r % 32 : r);
      const long wr = min(c, p.N - 1) + (GLU && r >= 32 ? p.N : 0);
      ws[r][x % 16] = k < p.K ? ldf(w + wr * p.K + k) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 16; s += 4) {
      const float b = ws[wave * 16 + i][s + g];
#pragma unroll
      for (int m = 0; m < 2; ++m)
        acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(xs[m * 16 + i][s + g], b, acc[m],
                                                      0, 0, 0);
    }
  }
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) cs[m * 16 + 4 * g + r][wave * 16 + i] = acc[m][r];
  __syncthreads();
  for (int x = tid; x < 32 * BN; x += 256) {
    const int r = x / BN, c = x % BN;
    if (r >= cnt || n0 + c >= p.N) continue;
    float v = GLU ? clamped_glu(cs[r][c], cs[r][32 + c], p) : cs[r][c];
    if constexpr (ACT == RELU2_ACT) v = v > 0.f ? v * v : 0.f;
    stf((T*)p.y + (long)(row0 + r) * p.N + n0 + c, v);
  }
}

// bf16, K a multiple of 64: TM rows x TB weight rows (GLU: half gate, half up), K in
// steps of 64 through an NS-deep ring of LDS stages filled by direct-to-LDS
// loads. A stage's 16-byte units are XOR-swizzled by row so that fragment reads
// are free of bank conflicts. A wave's columns hold gate and up of the same
// outputs, so the activation is register to register.
#define GK 64

template <int TM, int TB, int NS, int NTHR, int ACT>
__global__ __launch_bounds__(NTHR) void grouped_bf16_kernel(GroupArgs p) {
  constexpr bool GLU = ACT == GLU_ACT;
  const int* tb = p.table + blockIdx.y * 3;
  const int e = tb[0];
  if (e < 0) return;
  constexpr int MW = TM >= 64 ? 2 : 1;        // waves along rows
  constexpr int NW = NTHR / 64 / MW;          // waves along columns
  constexpr int WM = TM / MW, WN = TB / NW;   // a wave's tile
  constexpr int MI = WM / 16, NI = WN / 16;
  constexpr int LA = TM * 8 / NTHR, LB = TB * 8 / NTHR;  // loads per thread
  constexpr int STAGE = (TM + TB) * GK * 2;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int row0 = tb[1], cnt = tb[2];
  const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
  const int i = lane & 15, g = lane >> 4;
  constexpr int BN = GLU ? TB / 2 : TB;
  const int n0 = blockIdx.x * BN;
  const int K = p.K;
  const bf16_t* w = (const bf16_t*)p.w + (long)e * (GLU ? 2 : 1) * p.N * K;

  // source of each 16-byte unit this thread fills (LDS is linear in the lane)
  const bf16_t* as[LA];
  const bf16_t* bs[LB];
#pragma unroll
  for (int x = 0; x < LA; ++x) {
    const int r = (tid + x * NTHR) >> 3, unit = (tid & 7) ^ (r & 7);
    const int src = row0 + min(r, cnt - 1);
    as[x] = (const bf16_t*)p.x + (long)(p.gather ? p.gather[src] : src) * K + unit * 8;
  }
#pragma unroll
  for (int x = 0; x < LB; ++x) {
    const int r = (tid + x * NTHR) >> 3, unit = (tid & 7) ^ (r & 7);
    long wr;
    if constexpr (GLU) {  // within a wave's columns: first half gate, second up
      const int q = r % WN, c = n0 + r / WN * (WN / 2) + q % (WN / 2);
      wr = min(c, p.N - 1) + (q >= WN / 2 ? p.N : 0);
    } else {
      wr = min(n0 + r, p.N - 1);
    }
    bs[x] = w + wr * K + unit * 8;
  }
  auto issue = [&](int c) {
    char* st = lds + (c % NS) * STAGE;
#pragma unroll
    for (int x = 0; x < LA; ++x)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(as[x] + (long)c * GK),
          (__attribute__((address_space(3))) void*)(st + (tid + x * NTHR) * 16), 16, 0, 0);
#pragma unroll
    for (int x = 0; x < LB; ++x)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(bs[x] + (long)c * GK),
          (__attribute__((address_space(3))) void*)(st + TM * GK * 2 + (tid + x * NTHR) * 16),
          16, 0, 0);
  };
  floatx4 acc[MI][NI];
#pragma unroll
  for (int m = 0; m < MI; ++m)
#pragma unroll
    for (int n = 0; n < NI; ++n) acc[m][n] = floatx4{0.f, 0.f, 0.f, 0.f};

  const int nc = K / GK;
  const int wm = wave / NW * WM, wn = wave % NW * WN;
#pragma unroll
  for (int c = 0; c < NS - 1; ++c)
    if (c < nc) issue(c);
  for (int c = 0; c < nc; ++c) {
    // stage c has landed when at most the NS - 2 later ones are in flight. A
    // plain s_barrier: __syncthreads would drain the later stages as well.
    if (c + NS - 1 <= nc)
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier"
                   ::"n"((NS - 2) * (LA + LB)) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (c + NS - 1 < nc) issue(c + NS - 1);
    const char* xa = lds + (c % NS) * STAGE;
    const char* wb = xa + TM * GK * 2;
#pragma unroll
    for (int s = 0; s < GK / 32; ++s) {
      mfrag a[MI], b[NI];
#pragma unroll
      for (int m = 0; m < MI; ++m) {
        const int r = wm + m * 16 + i;
        a[m].s = *reinterpret_cast<const shortx8*>(xa + r * 128 + (((s * 4 + g) ^ (r & 7)) << 4));
      }
#pragma unroll
      for (int n = 0; n < NI; ++n) {
        const int r = wn + n * 16 + i;
        b[n].s = *reinterpret_cast<const shortx8*>(wb + r * 128 + (((s * 4 + g) ^ (r & 7)) << 4));
      }
#pragma unroll
      for (int m = 0; m < MI; ++m)
#pragma unroll
        for (int n = 0; n < NI; ++n)
          acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m].v, b[n].v, acc[m][n],
                                                              0, 0, 0);
    }
  }
  bf16_t* y = (bf16_t*)p.y;
  constexpr int NO = GLU ? NI / 2 : NI;
#pragma unroll
  for (int m = 0; m < MI; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = wm + m * 16 + 4 * g + r;
      if (row >= cnt) continue;
#pragma unroll
      for (int n = 0; n < NO; ++n) {
        const int c = n0 + (GLU ? wn / 2 : wn) + n * 16 + i;
        if (c >= p.N) continue;
        float v = GLU ? clamped_glu(acc[m][n][r], acc[m][n + (GLU ? NO : 0)][r], p)
                      : acc[m][n][r];
        if constexpr (ACT == RELU2_ACT) v = v > 0.f ? v * v : 0.f;
        y[(long)(row0 + row) * p.N + c] = f32_to_bf16(v);
      }
    }
}

// The same for well filled experts and for products of many rows: up to 256 rows x 256 weight
// rows, eight waves of half the rows and 64 columns each, two stages of 64 of K. While the
// products of 32 of K run, the fragments of the next 32 are read between them; a stage is
// requested as soon as all have read its predecessor but one, a stage's products ahead, and
// costs one barrier. Rows of a stage are whole cache lines (half lines halve what the L2
// delivers, 72 and 136 GB/s a CU). A fifth slot of the ring lets w, which comes from further
// away than x, be asked for two stages ahead; requests go out between the first products of
// a half, where they cost the least.
// The bound is power: the matrix cores are busy nine tenths of a stage, at the 1.7 GHz that
// this load leaves (8192^3 1.52 PFLOP/s, the stages alone 1.60; products of 32 x 32 leave 1.55
// GHz). What is left are the ends of tiles, and rows that are not there. So a workgroup stays
// on its CU and takes a tile of every round, with the next tile's first two stages on their
// way while it finishes one; outputs leave as whole lines and past the caches (4096 x 28672 x
// 1024: 250 us, with 32-byte pieces from a new workgroup for each tile, and now 198; 27700 x
// 2304 x 768: 123 and 85); and a tile has as many rows as its table says, 32 of them a step,
// of which a wave multiplies half (6176 x 4096 x 14336: 575 and 531).
template <int ACT>
__global__ __launch_bounds__(512) void grouped_large_kernel(GroupArgs p, int tiles, int cols) {
#ifdef __HIP_DEVICE_COMPILE__  // (the host pass does not know a buffer's descriptor)
  constexpr bool GLU = ACT == GLU_ACT || ACT == SILU_ACT;
  constexpr int BN = GLU ? 128 : 256, SLOT = 256 * GK * 2, RING = 5 * SLOT, L = 4;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int K = p.K, steps = K / GK;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int wr = wave / 4 * 16, wn = wave % 4 * 64;  // rows 32 m + wr + 0..15, columns

  // The tile that is multiplied and the next. A round's tiles lie in bands of up to eight row
  // tiles, down and then across; an XCD takes neighbours, which share rows and columns in
  // its L2.
  const int nt = p.table ? __builtin_amdgcn_readfirstlane(p.table[tiles * 3]) : tiles;
  const int bands = (nt + 7) / 8, high = bands ? (nt + bands - 1) / bands : 1;
  int e = 0, row0 = 0, cnt = 0, n0 = 0, row_now = 0, cnt_now = 0, n_now = 0;
  auto locate = [&](int round) {  // false: there is none
    const long left = (long)nt * cols - round * 256L;
    const int share = (int)(min(left, 256L) + 7) / 8, at = blockIdx.x / 8;
    if (left <= 0 || at >= share || (int)(blockIdx.x % 8) * share + at >= left) return false;
    const unsigned v = round * 256 + blockIdx.x % 8 * share + at, band = v / (high * cols);
    const unsigned in = v - band * high * cols, h = min(high, nt - (int)band * high);
    const int rt = band * high + in % h;
    n0 = in / h * BN;
    if (p.table) {
      e = p.table[rt * 3];
      row0 = p.table[rt * 3 + 1];
      cnt = p.table[rt * 3 + 2];
    } else {
      const long parts = (p.rows + 31) / 32;
      row0 = (int)(rt * parts / nt) * 32;
      cnt = min((int)((rt + 1) * parts / nt) * 32, p.rows) - row0;
    }
    return true;
  };
  if (!locate(0)) return;

  const unsigned wbytes = (unsigned)((GLU ? 2 : 1) * p.N) * (unsigned)(K * 2);
  auto weights = [&] {
    return __builtin_amdgcn_make_buffer_rsrc((char*)p.w + e * (long)wbytes, 0, wbytes, 0x00027000);
  };
  // x from the tile's first row on, where its rows are picked from its first
  const unsigned xrow = (p.ldx ? p.ldx : K) * 2;
  auto inputs = [&] {
    return __builtin_amdgcn_make_buffer_rsrc(
        (char*)p.x + (p.gather ? 0 : row0 * (long)xrow), 0,
        (unsigned)((p.gather ? p.rows : cnt) - 1) * xrow + (unsigned)(K * 2), 0x00027000);
  };
  auto wres = weights(), xres = inputs();
  // offsets of the 16-byte units this thread fills: rows of x, then of w
  unsigned xo[L], wo[L];
  auto aim = [&] {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // nothing of this is kept through the products
    const int unit = (tid & 7) ^ (tid >> 3 & 7);
#pragma unroll
    for (int l = 0; l < L; ++l) {
      const int r = (tid >> 3) + l * 64, row = min(r, cnt - 1);
      xo[l] = (unsigned)(p.gather ? p.gather[row0 + row] : row) * xrow + unit * 16;
      int wrow;
      if constexpr (GLU)  // of a wave's 64 columns half are gate's, half up's
        wrow = min(n0 + l * 32 + (r & 31), p.N - 1) + (r >> 5 & 1) * p.N;
      else
        wrow = min(n0 + r, p.N - 1);
      wo[l] = (unsigned)wrow * (unsigned)(K * 2) + unit * 16;
    }
    wres = weights(), xres = inputs();
  };
  aim();
  // the ring's slots take w's and x's blocks of 64 of K in turn
  int to = 0;
  auto request_w = [&](int stage, int l) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        wres, (lptr_t)(lds + to + (l * 512 + wave * WAVE) * 16), 16, wo[l], stage * (GK * 2), 0, 0);
  };
  auto request_x = [&](int stage, int l) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        xres, (lptr_t)(lds + to + (l * 512 + wave * WAVE) * 16), 16, xo[l], stage * (GK * 2), 0, 0);
  };
  auto advance = [&] { to = to == RING - SLOT ? 0 : to + SLOT; };
  int at_w = 0;  // slot of w's block of this stage
  auto next = [&] { at_w = at_w >= 3 * SLOT ? at_w - 3 * SLOT : at_w + 2 * SLOT; };
#pragma unroll
  for (int x = 0; x < 4; ++x) {
#pragma unroll
    for (int l = 0; l < L; ++l)
      if (x % 2) request_x(x / 2, l);
      else request_w(x / 2, l);
    advance();
  }
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * L) : "memory");

  using FIRST = std::integral_constant<int, 0>;
  using SECOND = std::integral_constant<int, 1>;
  // a tile of up to 32 MI rows, whose first stage has landed
  auto tile = [&](auto MI_, bool more) {
    constexpr int MI = decltype(MI_)::value;
    int lane = threadIdx.x % WAVE;
    asm volatile("" : "+v"(lane));  // the same
    const int i = lane & 15, g = lane >> 4;
    const int unit = (g ^ (i & 7)) * 16;  // of the first 32 of K; of the second ^ 64
    const int xa = (wr + i) * 128, wb = (wn + i) * 128;
    frag_u a[2][MI], b[2][4];
    auto read_b = [&](auto HALF, int n) {
      constexpr int h = decltype(HALF)::value;
      b[h][n].s =
          *reinterpret_cast<const shortx8*>(lds + (unit ^ h * 64) + at_w + wb + n * 2048);
    };
    auto read_a = [&](auto HALF, int m) {
      constexpr int h = decltype(HALF)::value;
      const int behind = at_w == RING - SLOT ? 0 : at_w + SLOT;
      a[h][m].s =
          *reinterpret_cast<const shortx8*>(lds + (unit ^ h * 64) + behind + xa + m * 4096);
    };
#pragma unroll
    for (int n = 0; n < 4; ++n) read_b(FIRST{}, n);
#pragma unroll
    for (int m = 0; m < MI; ++m) read_a(FIRST{}, m);
    floatx4 acc[MI][4];
#pragma unroll
    for (int m = 0; m < MI; ++m)
#pragma unroll
      for (int n = 0; n < 4; ++n) acc[m][n] = floatx4{0.f, 0.f, 0.f, 0.f};
    // The products of a half; between them ``COUNT`` requests of the block (first w's, then
    // x's) of ``stage`` and, with AHEAD, the next half's fragments, in this order.
    auto half = [&](auto HALF, auto COUNT, int stage, auto AHEAD) {
      constexpr int h = decltype(HALF)::value, count = decltype(COUNT)::value;
      constexpr int reads = decltype(AHEAD)::value ? 4 + MI : 0;
      using OTHER = std::integral_constant<int, 1 - h>;
#pragma unroll
      for (int l = 0; l < count; ++l)
        if (h) request_x(stage, l);
        else request_w(stage, l);
      advance();
      if constexpr (reads > 0) {
#pragma unroll
        for (int n = 0; n < 4; ++n) read_b(OTHER{}, n);
#pragma unroll
        for (int m = 0; m < MI; ++m) read_a(OTHER{}, m);
      }
#pragma unroll
      for (int m = 0; m < MI; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n)
          acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[h][n].v, a[h][m].v, acc[m][n],
                                                              0, 0, 0);
#pragma unroll
      for (int l = 0; l < count; ++l) {
        __builtin_amdgcn_sched_group_barrier(0x008, MI > 5 ? 2 : 1, 0);  // products
        __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);               // a request
      }
#pragma unroll
      for (int x = 0; x < reads; ++x) {
        if (MI > 3 || x % 2) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // a read
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    // The next stage has landed, which is all that was asked for but the last block of w,
    // and all have read this one.
    auto middle = [&] {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(L) : "memory");
      next();
    };
    using ALL = std::integral_constant<int, L>;
    using ROWS = std::integral_constant<int, (MI + 1) / 2>;  // requests that hold x's rows
    for (int s = 2; s < steps; ++s) {
      half(FIRST{}, ALL{}, s, std::true_type{});
      middle();
      half(SECOND{}, ROWS{}, s, std::true_type{});
    }
    if (more) aim();  // else the same two stages again, for nothing
    half(FIRST{}, ALL{}, 0, std::true_type{});
    middle();
    half(SECOND{}, ALL{}, 0, std::true_type{});
    half(FIRST{}, ALL{}, 1, std::true_type{});
    middle();
    half(SECOND{}, ALL{}, 1, std::false_type{});

    // A lane has four outputs of a row side by side. They become whole lines (GLU: halves of
    // them) in the ring's free slot, in those parts of it that this wave's own requests fill,
    // so that nobody waits for another; 16-byte units are xored by row.
    constexpr int NO = GLU ? 2 : 4, UNITS = NO * 2, ROWS_ = 64 / UNITS;  // of a part of 1 KB
    constexpr int ONCE = GLU ? 4 : 2;  // m at once
    char* const part = lds + to + wave * 1024;
    const int lr = (int)((unsigned)lane / UNITS), lu = (int)((unsigned)lane % UNITS);
    const int c = n_now + (GLU ? wn / 2 : wn) + lu * 8;
    bf16_t* const dst = (bf16_t*)p.y + (long)(row_now + wr + lr) * p.N + c;
#pragma unroll
    for (int m0 = 0; m0 < MI; m0 += ONCE) {
#pragma unroll
      for (int m = m0; m < (m0 + ONCE < MI ? m0 + ONCE : MI); ++m) {
        const int r = (m - m0) * 16 + i;
#pragma unroll
        for (int n = 0; n < NO; ++n) {
          float v[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float x = acc[m][n][q], up = acc[m][n + (GLU ? NO : 0)][q];
            v[q] = ACT == SILU_ACT ? silu_glu(x, up) : GLU ? clamped_glu<true>(x, up, p) : x;
            if constexpr (ACT == RELU2_ACT) v[q] = v[q] > 0.f ? v[q] * v[q] : 0.f;
          }
          const int u = (n * 2 + (g >> 1)) ^ (r & (UNITS - 1));
          *reinterpret_cast<u64b*>(part + r / ROWS_ * 8192 + r % ROWS_ * (UNITS * 16) + u * 16 +
                                   (g & 1) * 8) =
              (u64b)cvt2_bf16(v[2], v[3]) << 32 | cvt2_bf16(v[0], v[1]);
        }
      }
      shortx8 v[4];
#pragma unroll
      for (int t = 0; t < 4; ++t)
        v[t] = *reinterpret_cast<const shortx8*>(part + t * 8192 + lr * (UNITS * 16) +
                                                 ((lu ^ lr) & (UNITS - 1)) * 16);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int at = (m0 + t * ROWS_ / 16) * 32 + t * ROWS_ % 16;
        if (at + wr + lr < cnt_now && c < p.N)
          __builtin_nontemporal_store(v[t], reinterpret_cast<shortx8*>(dst + (long)at * p.N));
      }
      asm volatile("" ::: "memory");
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // before the slot is asked to be filled
    __builtin_amdgcn_sched_barrier(0);
  };

  bool more = true;
  for (int round = 1; more; ++round) {
    row_now = row0, cnt_now = cnt, n_now = n0;
    more = locate(round);
    const int parts = (cnt_now + 31) / 32;
    if (parts <= 2) tile(std::integral_constant<int, 2>{}, more);
    else if (parts <= 4) tile(std::integral_constant<int, 4>{}, more);
    else if (parts == 5) tile(std::integral_constant<int, 5>{}, more);
    else if (parts == 6) tile(std::integral_constant<int, 6>{}, more);
    else if (parts == 7) tile(std::integral_constant<int, 7>{}, more);
    else tile(std::integral_constant<int, 8>{}, more);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // requests must not outlive the workgroup
#endif
}

template <int ACT>
static void grouped_large(const GroupArgs& p, int tiles) {
  constexpr int BN = ACT == GLU_ACT || ACT == SILU_ACT ? 128 : 256, lds = 5 * 256 * GK * 2;
  auto kern = grouped_large_kernel<ACT>;
  static const hipError_t once = hipFuncSetAttribute(
      (const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  (void)once;
  hipLaunchKernelGGL(kern, dim3(256), dim3(512), lds, CUR_STREAM, p, tiles, (p.N + BN - 1) / BN);
}

template <int TM, int TB, int NS, int NTHR, int ACT>
static void grouped_bf16(const GroupArgs& p, int tiles) {
  constexpr int BN = ACT == GLU_ACT ? TB / 2 : TB;
  constexpr int lds = NS * (TM + TB) * GK * 2;
  auto kern = grouped_bf16_kernel<TM, TB, NS, NTHR, ACT>;
  if (lds > 64 * 1024) {
    static const hipError_t once = hipFuncSetAttribute(
        (const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    (void)once;
  }
  hipLaunchKernelGGL(kern, dim3((p.N + BN - 1) / BN, tiles), dim3(NTHR), lds, CUR_STREAM, p);
}

template <int ACT>
static void grouped(const GroupArgs& p, bool bf16, int tiles, int TM, long busy) {
  constexpr bool GLU = ACT == GLU_ACT;
  if (bf16 && p.K % GK == 0) {
    const long blocks = (p.N + (GLU ? 63 : 127)) / (GLU ? 64 : 128) * busy;
    if (TM == 256 && ACT == GLU_ACT && p.silu) grouped_large<SILU_ACT>(p, tiles);
    else if (TM == 256) grouped_large<ACT>(p, tiles);
    else if (TM == 128) grouped_bf16<128, 128, 2, 256, ACT>(p, tiles);
    else if (TM == 64) grouped_bf16<64, 128, 3, 256, ACT>(p, tiles);
    // few rows: the weights' stream counts. Two workgroups per CU with four
    // stages each, or one with seven where there are not enough for two
    else if (blocks >= 512) grouped_bf16<32, 128, 4, 256, ACT>(p, tiles);
    else grouped_bf16<32, 128, 7, 256, ACT>(p, tiles);
    return;
  }
  TORCH_CHECK(TM == 32);
  const dim3 grid((p.N + (GLU ? 31 : 63)) / (GLU ? 32 : 64), tiles);
  if (bf16)
    hipLaunchKernelGGL((grouped_any_kernel<bf16_t, ACT>), grid, dim3(256), 0, CUR_STREAM, p);
  else
    hipLaunchKernelGGL((grouped_any_kernel<float, ACT>), grid, dim3(256), 0, CUR_STREAM, p);
}

bool large_takes(long N, long K);

// 16-byte loads straight to LDS can read it
static bool unit_aligned(const torch::Tensor& t) { return (uintptr_t)t.data_ptr() % 16 == 0; }

template <int ACT>
static std::vector<torch::Tensor> experts(torch::Tensor h, const torch::Tensor& sel,
                                          torch::Tensor w_up, torch::Tensor w_dn,
                                          double limit, double alpha, double shift,
                                          bool silu = false) {
  TORCH_CHECK(h.is_cuda() && h.dim() == 2 && h.is_contiguous() && sel.is_contiguous() &&
              sel.dtype() == torch::kInt32 && sel.size(0) == h.size(0));
  const long T_ = h.size(0), W = h.size(1), top = sel.size(1), A = T_ * top;
  const long E = w_up.size(0), F = w_up.size(1) / (ACT == GLU_ACT ? 2 : 1);
  TORCH_CHECK(w_up.is_contiguous() && w_dn.is_contiguous() && w_up.dtype() == h.dtype() &&
              w_dn.dtype() == h.dtype() && w_up.size(2) == W && w_dn.size(0) == E &&
              w_dn.size(1) == W && w_dn.size(2) == F && E <= MAX_EXPERTS);
  auto i32 = h.options().dtype(torch::kInt32);
  auto y = torch::empty({A, W}, h.options()), place = torch::empty({T_, top}, i32);
  if (A == 0) return {y, place};
  const bool bf16 = h.dtype() == torch::kBFloat16;
  // Row tile, us of tiles of 32, 64 and 256 (both products, uneven experts). While rows are few
  // the weights' stream counts, and the 32-row tile has the longest ring: it is the best up to
  // 48 rows an expert where the down product has fewer than 256 blocks (8 experts of 2048 x 8192,
  // 30 rows on average 177 196 239, 46 rows 213 197 246), up to 26 where it has 1024 and more (64
  // of 2048 x 1408, 22 rows 222 234 241, 34 rows 249 235 243), up to 16 between (8 of 4096 x
  // 14336, 12 rows 522 535 555, 22 rows 630 533 563; 16 of 2048 x 5632, squared relu, 18 rows 167
  // 144 171). The 256-row tile wants blocks for a good part of the chip: large weights 40 rows on
  // (8 of 4096 x 14336, 40 rows 738 618 588; 512 of 4096 x 1536, 46 rows 4114 3659 3556; but 8 of
  // 2048 x 8192, 96 rows (112 blocks) 316 224 251, 160 rows (144) 446 298 267), less than 2^22 of
  // them an expert 52 (128 of 2048 x 768, 46 rows 322 270 277, 56 rows 350 288 284), less than 2^20
  // 26 (64 of 1024 x 512, 30 rows 48 55 51; 512, 50 rows 400 368 356; but 16, 160 rows (144 blocks)
  // 47 32 37). Over 672 sizes the choice costs 0.7% beside the fastest. 128 rows are left to sizes
  // that the 256-row tile has no form for.
  const bool matrix = bf16 && W % GK == 0 && F % GK == 0;
  for (auto* t : {&h, &w_up, &w_dn})
    if (bf16 && !unit_aligned(*t)) *t = t->clone();
  const bool large = matrix && large_takes(2 * F, W) && large_takes(W, F) && T_ * W < 1l << 30;
  const bool small = W * F < 1l << 20;
  const long cols = ACT == GLU_ACT ? 128 : 256;
  const long wide = std::min((F + cols - 1) / cols, (W + 255) / 256);
  const long blocks = (A / 128 + E) * wide;
  const long down = (W + 127) / 128 * std::min(E, A);
  const long few = down < 256 ? 48 : down < 1024 ? 16 : 26;
  const long many = small ? 26 : W * F < 1l << 22 ? 52 : 40;
  const int TM = !matrix                                                      ? 32
                 : large && A >= many * E && blocks >= (small ? 170 : 144)    ? 256
                 : A < few * E                                                ? 32
                 : large || A < 160 * E                                       ? 64 : 128;
  const int tiles = (int)(A / (TM == 256 ? 128 : TM) + std::min(E, A));
  auto token = torch::empty({A}, i32), table = torch::empty({2, tiles + 1, 3}, i32);
  auto act = torch::empty({A, F}, h.options());
  hipLaunchKernelGGL(moe_sort_kernel, dim3(1), dim3(1024), 0, CUR_STREAM,
                     sel.data_ptr<int>(), (int)A, (int)E, (int)top, TM, tiles,
                     (int)((F + cols - 1) / cols), (int)((W + 255) / 256),
                     place.data_ptr<int>(), token.data_ptr<int>(), table.data_ptr<int>());
  GroupArgs p = {h.data_ptr(), token.data_ptr<int>(), w_up.data_ptr(), act.data_ptr(),
                 table.data_ptr<int>(), (int)F, (int)W, (float)limit, (float)alpha,
                 (float)shift, (int)T_};
  // silu_mul's exponential, off by 3.9e-6 where expf is by 1.75e-7, only where rows are many
  // enough for the activation to show: 8 experts of 4096 x 14336, two each, 38 to 80 rows an
  // expert 562 to 590 us and with expf 0.2 to 0.7% more, 150 to 2000 rows 1.2 to 2.2%.
  p.silu = silu && A >= 80 * E && std::max(std::min(E, A), A / 256) * wide >= 96;
  grouped<ACT>(p, bf16, tiles, TM, std::min(E, A));
  p.x = act.data_ptr();
  p.rows = (int)A;
  p.gather = nullptr;
  p.w = w_dn.data_ptr();
  p.y = y.data_ptr();
  if (TM == 256) p.table += (tiles + 1) * 3;
  p.N = W;
  p.K = F;
  grouped<NO_ACT>(p, bf16, tiles, TM, std::min(E, A));
  HIP_CHECK_KERNEL();
  return {y, place};
}

std::vector<torch::Tensor> moe_clamped_glu(torch::Tensor h, torch::Tensor sel,
                                           torch::Tensor w_gu, torch::Tensor w_dn,
                                           double limit, double alpha, double shift) {
  return experts<GLU_ACT>(h, sel, w_gu, w_dn, limit, alpha, shift);
}

// silu(gate) up
std::vector<torch::Tensor> moe_silu_glu(torch::Tensor h, torch::Tensor sel, torch::Tensor w_gu,
                                        torch::Tensor w_dn) {
  return experts<GLU_ACT>(h, sel, w_gu, w_dn, INFINITY, 1.0, 0.0, true);
}

// Into how many tiles of at most 256 rows, and ``cols`` columns, a product is cut, evenly
static int row_tiles(long rows, long cols) {
  const long parts = (rows + 31) / 32, least = (parts + 7) / 8;
  long best = least;
  float low = 0;
  for (long n = least; n <= std::min(parts, least < 8 ? 8 * least : 2 * least); ++n) {
    const float time = rounds_time(n * cols, (float)parts / n, (int)((parts + n - 1) / n));
    if (n == least || time < low) low = time, best = n;
  }
  return (int)best;
}

// Whether the kernel of 256-row tiles has a form for the product: whole pieces of 16 bytes of
// an output row, two stages of K, w and a tile's rows of x (picked ones: all) within the 31
// bits of their offsets.
bool large_takes(long N, long K) {
  return K % GK == 0 && K >= 2 * GK && K < 1l << 22 && N % 8 == 0 && N * K < 1l << 30;
}

// x [T, K], whose rows may be strided, @ w^T, with ``silu`` silu(gate) * up of the products
// with w's halves, of a size that large_takes
torch::Tensor many_rows(torch::Tensor x, torch::Tensor w, bool silu) {
  TORCH_CHECK(x.is_cuda() && w.is_cuda() && x.dtype() == torch::kBFloat16 &&
                  w.dtype() == torch::kBFloat16 && w.is_contiguous() && unit_aligned(w) &&
                  x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1) &&
                  w.size(0) % (silu ? 16 : 8) == 0 && large_takes(w.size(0), x.size(1)),
              "bf16 on the GPU, K a multiple of ", GK, " from ", 2 * GK, " on, whole pieces of 8 "
              "outputs");
  const long T_ = x.size(0), K = x.size(1), N = w.size(0) / (silu ? 2 : 1);
  auto y = torch::empty({T_, N}, x.options());
  if (T_ == 0 || N == 0) return y;
  if (!unit_aligned(x) || x.stride(1) != 1 ||
      (T_ > 1 && (x.stride(0) % 8 || x.stride(0) < K || x.stride(0) >= 1l << 22)))
    x = x.clone(at::MemoryFormat::Contiguous);
  GroupArgs p = {x.data_ptr(), nullptr, w.data_ptr(), y.data_ptr(), nullptr, (int)N,
                 (int)K, INFINITY, 1.f, 0.f, (int)T_};
  if (T_ > 1) p.ldx = (int)x.stride(0);
  const int tiles = row_tiles(T_, silu ? (N + 127) / 128 : (N + 255) / 256);
  if (silu) grouped_large<SILU_ACT>(p, tiles);
  else grouped_large<NO_ACT>(p, tiles);
  HIP_CHECK_KERNEL();
  return y;
}

std::vector<torch::Tensor> moe_relu2(torch::Tensor h, torch::Tensor sel, torch::Tensor w_up,
                                     torch::Tensor w_dn) {
  return experts<RELU2_ACT>(h, sel, w_up, w_dn, 0.0, 0.0, 0.0);
}

// ------------------------------------------------------------------ combine

// Every token's expert rows, weighted and summed in fp32; a thread owns 8 columns. Bound
// by memory: 1580 tokens of 4096 with two experts each, 39 MB.
__global__ __launch_bounds__(256) void moe_combine_kernel(
    const bf16_t* __restrict__ y, const int* __restrict__ place,
    const float* __restrict__ gate, bf16_t* __restrict__ out, long T_, int W, int top) {
  const long x = blockIdx.x * 256L + threadIdx.x;
  const int w8 = W / 8;
  const long t = x / w8;
  if (t >= T_) return;
  const int c = x % w8 * 8;
  float acc[8] = {};
  for (int k = 0; k < top; ++k) {
    const float g = gate[t * top + k];
    const shortx8 v = *reinterpret_cast<const shortx8*>(y + (long)place[t * top + k] * W + c);
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] += g * bf16_to_f32((unsigned short)v[j]);
  }
  shortx8 r;
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = (short)f32_to_bf16(acc[j]);
  *reinterpret_cast<shortx8*>(out + t * W + c) = r;
}

// y [T * top, W] rows of the sorted batch, place and gate [T, top] -> [T, W]
torch::Tensor moe_combine(torch::Tensor y, torch::Tensor place, torch::Tensor gate) {
  TORCH_CHECK(y.is_cuda() && y.dtype() == torch::kBFloat16 && y.is_contiguous() &&
              place.is_contiguous() && place.dtype() == torch::kInt32 &&
              gate.is_contiguous() && gate.dtype() == torch::kFloat32 &&
              place.sizes() == gate.sizes() && y.size(0) == place.numel());
  const long T_ = place.size(0), W = y.size(1);
  TORCH_CHECK(W % 8 == 0, "rows of a multiple of 8");
  auto out = torch::empty({T_, W}, y.options());
  if (T_ == 0) return out;
  hipLaunchKernelGGL(moe_combine_kernel, dim3((T_ * (W / 8) + 255) / 256), dim3(256), 0,
                     CUR_STREAM, (const bf16_t*)y.data_ptr(), place.data_ptr<int>(),
                     gate.data_ptr<float>(), (bf16_t*)out.data_ptr(), T_, (int)W,
                     (int)place.size(1));
  HIP_CHECK_KERNEL();
  return out;
}
