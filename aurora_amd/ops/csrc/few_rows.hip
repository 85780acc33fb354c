// Products of few rows for gfx950: out[M <= 128, N] = x[M, K] @ W[N, K]^T, what a decoding
// step does with every dense weight, and silu(gate) * up of such products.
//
// Bound by reading W once. A workgroup takes 64 rows of W (96 to 128 for the wide forms) and
// all rows of x, in steps of 64 of K through a ring of LDS stages that direct-to-LDS loads fill
// several steps ahead: two workgroups of 72 to 80 KB fit a CU and have 48 to 80 KB of W
// under way. A wave multiplies 16 rows of W with all of x, or from 33 rows of x on 32 with
// half of it, which takes less from LDS: a lane ends with four outputs that lie side by side.
// Reading W straight into fragments instead, with K split over the waves of a workgroup and no
// LDS, came to the same at one row and lost at 16 and more
// (x is then read as often as W's tiles of 16 rows: 28672 x 4096, 32 rows, 86 us).
//
// Few tiles of W leave the chip idle, so K is cut into parts as well (``parts_of``). Their
// fp32 sums are added by whatever reads the product next (norm or rotation, 0.1 to 0.7 us)
// or by a kernel of their own (2.4 to 4.7 us).
//
// Cold weights in a graph, with the parts not yet added; before are the kernel of shallow
// stages that this replaced, its combining kernel included, or the library's from 65 rows:
//   N x K          rows: 1            23           64           96           128
//   4096 x 4096    14.4 ->  8.0   14.2 ->  8.9  15.6 -> 10.0  22.2 -> 11.5  24.4 -> 13.6 us
//   6144 x 4096    15.4 -> 12.3   16.2 -> 13.4  20.1 -> 16.3  23.3 -> 18.7  25.8 -> 21.6
//   4096 x 14336   28.2 -> 23.0   29.0 -> 24.1  33.5 -> 27.4  52.3 -> 32.1  55.5 -> 38.1
//   2048 x 2048     8.3 ->  3.8    9.0 ->  4.0  10.4 ->  5.5   8.5 ->  6.4   8.5 ->  7.2
//   2048 x 8192    15.1 ->  8.6   15.8 ->  9.3  16.7 -> 10.4  25.0 -> 12.2  25.2 -> 14.4
//   28672 x 4096, with silu (two kernels before)
//                  66.3 -> 48.5   58.2 -> 48.0  56.8 -> 53.3  60.1 -> 56.1  62.8 -> 59.3
// (4096 x 14336 is 21 us at the 5.6 TB/s of a large read, 28672 x 4096 42 us). What is left
// at 64 rows and more is x on its way to every CU. Asking for W ahead of the product, from
// workgroups beside those of the norm before it, brings nothing (4096 x 14336, norm, 28672 x
// 4096, 23 rows: 73.5 us, and with 4 to 29 MB asked for 73.2 to 77): what comes from
// memory and what lies in the cache before it take the same way.
//
// Up to 1000 rows come in blocks of 64, 96 or 128 (``block_cut``), bound by the stages of the
// workgroups' tiles: 4096 x 4096, 140 and 512 rows, 18 and 28 us, the library's product 22 and 29.
#include "flash_tiles.h"
#include <torch/extension.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#define CUR_STREAM c10::hip::getCurrentHIPStream().stream()

#define FEW_K 64      // K of a stage: eight 16-byte units a row, XOR-swizzled by row
#define FEW_MOST 128  // rows of x

// This wave's loads but the last L have landed, its reads are done, and so for all waves.
template <int L>
DEVINL void await_stage() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(L) : "memory");
}

// WN rows of W, 16 MT rows of x, NS stages. SILU: W is gate's N rows, then up's; a wave's 16
// rows are 8 of each. Outputs are bf16, or with ``part`` sums over ``span`` of K; with both they
// go to ``part``, rounded to bf16 first. ROUTER: a workgroup y of Y takes every Y-th step and keeps
// the sums of its steps' two halves apart, parts 2 y and 2 y + 1; z are blocks of 16 MT rows of x.
// A wave's tiles of 16 are RT of W by MW of x. (2 by half of x instead of 1 by all: 64 wide 0.4%
// faster at 33 to 64 rows, 2.2% at 128, means of 18 weights of 16 MB and more.)
// (Tiles of one part of K side by side on an XCD, so that its L2 reads that part of x alone:
// products by themselves 1% faster, steps of 1 to 96 rows of whole models up to 1.5% slower.)
template <int WN, int MT, int NS, bool SILU, bool ROUTER = false>
__global__ __launch_bounds__(WN * 4) void few_rows_kernel(
    const unsigned short* x, const unsigned short* w, unsigned short* out, float* part, int M,
    int N, int K, int span, long ldx) {
  constexpr int NT = WN * 4;
  constexpr int RT = MT >= 4 && WN % 32 == 0 ? 2 : 1, MW = MT / RT, ACROSS = WN / 16 / RT;
  constexpr int L = (WN * 8 + MT * 128 + NT - 1) / NT;  // loads of a thread per stage
  constexpr int STAGE = L * NT * 16;
  __shared__ __attribute__((aligned(16))) char lds[NS * STAGE];
  const int tid = threadIdx.x, lane = tid % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int at = lane & 15, g = lane >> 4;
  const int r0 = wave % ACROSS * RT * 16, x0 = wave / ACROSS * MW * 16;
  const int n0 = blockIdx.x * (SILU ? WN / 2 : WN);
  const int k0 = blockIdx.y * (ROUTER ? FEW_K : span), m0 = blockIdx.z * 16 * MT;
  const int stride = ROUTER ? gridDim.y * FEW_K : FEW_K;
  const int steps = ROUTER ? max(K - k0 + stride - 1, 0) / stride
                           : (min(K, k0 + span) - k0) / FEW_K;
  const unsigned short* src[L];
#pragma unroll
  for (int l = 0; l < L; ++l) {
    const int r = (tid + l * NT) >> 3, unit = (tid & 7) ^ (r & 7);
    long row;  // rows past the end are the last again
    if (l >= WN * 8 / NT) row = min(m0 + r - WN, M - 1);
    else if constexpr (SILU) row = min(n0 + r / 16 * 8 + r % 8, N - 1) + (long)(r % 16 / 8) * N;
    else row = min(n0 + r, N - 1);
    src[l] = (l >= WN * 8 / NT ? x + row * ldx : w + row * K) + k0 + unit * 8;
  }
  auto issue = [&](int s) {
    char* stage = lds + s % NS * STAGE;
#pragma unroll
    for (int l = 0; l < L; ++l)
      __builtin_amdgcn_global_load_lds((gptr_t)(src[l] + (long)s * stride),
                                       (lptr_t)(stage + (l * NT + wave * WAVE) * 16), 16, 0, 0);
  };
  constexpr int SUMS = ROUTER ? 2 : 1;
  floatx4 acc[SUMS][RT][MW];
#pragma unroll
  for (int u = 0; u < SUMS * RT * MW; ++u)
    acc[u / (RT * MW)][u / MW % RT][u % MW] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto compute = [&](int s) {
    const char* stage = lds + s % NS * STAGE;
    frag_u wf[2][RT], xf[2][MW];  // all read before the first product: one latency a step
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int unit = ((h * 4 + g) ^ (at & 7)) * 16;
#pragma unroll
      for (int r = 0; r < RT; ++r)
        wf[h][r].s =
            *reinterpret_cast<const shortx8*>(stage + (r0 + r * 16 + at) * 128 + unit);
#pragma unroll
      for (int m = 0; m < MW; ++m)
        xf[h][m].s =
            *reinterpret_cast<const shortx8*>(stage + (WN + x0 + m * 16 + at) * 128 + unit);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int m = 0; m < MW; ++m)
          acc[h % SUMS][r][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              wf[h][r].v, xf[h][m].v, acc[h % SUMS][r][m], 0, 0, 0);
  };
  for (int s = 0; s < min(steps, NS - 1); ++s) issue(s);
  int s = 0;
  for (; s + NS - 1 < steps; ++s) {
    await_stage<(NS - 2) * L>();
    issue(s + NS - 1);  // over the stage before this, which all waves have left
    compute(s);
  }
  await_stage<0>();
  for (; s < steps; ++s) compute(s);

#pragma unroll
  for (int u = 0; u < SUMS * RT * MW; ++u) {
    const int m = u % MW, r = u / MW % RT, sum = u / (RT * MW);
    const int n = n0 + (SILU ? r0 / 2 + r * 8 + (g & 1) * 4 : r0 + r * 16 + g * 4);
    floatx4 y = acc[sum][r][m];
    if constexpr (SILU) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float up = __shfl_xor(y[j], 32, WAVE);
        y[j] = y[j] / (1.f + __expf(-y[j])) * up;
      }
      if (g >= 2) continue;
    }
    const int row = m0 + x0 + m * 16 + at;
    if (row >= M) continue;
    const bool whole = n + 4 <= N && N % 4 == 0;
    if (!SILU && part) {
      if (out) {  // as bf16 holds it
        const unsigned a = cvt2_bf16(y[0], y[1]), b = cvt2_bf16(y[2], y[3]);
        y = floatx4{__uint_as_float(a << 16), __uint_as_float(a & 0xffff0000u),
                    __uint_as_float(b << 16), __uint_as_float(b & 0xffff0000u)};
      }
      float* dst = part + ((long)(blockIdx.y * SUMS + sum) * M + row) * N + n;
      if (whole) *reinterpret_cast<floatx4*>(dst) = y;
      else
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (n + j < N) dst[j] = y[j];
    } else {
      unsigned short* dst = out + (long)row * N + n;
      if (whole)
        *reinterpret_cast<u64b*>(dst) =
            (u64b)cvt2_bf16(y[2], y[3]) << 32 | cvt2_bf16(y[0], y[1]);
      else
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (n + j < N) dst[j] = f32_to_bf16(y[j]);
    }
  }
}

// A wait for LDS alone: loads of W on their way to it stay under way.
DEVINL void meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

#define ROW_MOST 8192  // elements of the row below

// threads that norm the row, besides those of the product: wider rows want eight waves (4096
// wide, a layer 92.0 and 91.8 us, 2048 38.8 and 38.1, 1024 20.6 and 21.7)
constexpr int row_threads(int hv) { return hv > 1 ? 512 : 256; }

// The product of one row with the norm before it: x comes as S parts [S, K] to be added to the
// residual, as rmsnorm_residual does. Every workgroup norms the row for itself: four or eight
// waves of their own do that while four others have the first blocks of W on their way, and end.
// The first workgroup writes the new residual. HV: vectors of four of the row per 256 threads, S
// at most 16 / HV.
// Bound by W; what is saved is the norm's launch and its trip to memory, what it costs is the
// parts' way to every CU (64 KB). A layer of one row, its two norms before and in the products,
// cold weights: 4096 wide, 28672 and 6144 outputs, 95.9 and 91.8 us; 2048, 16384 and 3072, 41.0
// and 38.1; 1024, 8192 and 2048, 24.5 and 20.6. With the norm by the waves that load W (its
// loads are then waited for with W's) 93.7, 38.5 and 21.3. The two products alone with their
// norms, before and in them: 60.8 and 57.8, 27.2 and 24.4, 15.7 and 12.4; 8192 wide, 16384 and
// 10240 outputs, 106.0 and 102.2 (squares in the order of this kernel's threads: 57.9, 24.5, 12.2
// and 101.6, but a row in some hundred with an element off by its last bit).
template <int HV, bool SILU, int WN = 64>
__global__ __launch_bounds__(WN * 4 + row_threads(HV)) void one_row_kernel(
    const float* __restrict__ x, int S, const unsigned short* __restrict__ res,
    const unsigned short* __restrict__ weight, unsigned short* __restrict__ res_out, float eps,
    const unsigned short* __restrict__ w, unsigned short* __restrict__ out,
    float* __restrict__ part, int N, int K, int span) {
  constexpr int NT = WN * 4, NS = 7, L = 2, STAGE = WN * 128, RT = row_threads(HV);
  constexpr int PARTS = 16 / HV, V = HV * 256 / RT > 0 ? HV * 256 / RT : 1;
  // one array: of several the compiler waits for all loads under way before it reads one
  __shared__ __attribute__((aligned(16))) char lds[NS * STAGE + (V * RT * 8) + 64];
  auto* row = reinterpret_cast<unsigned short*>(lds + NS * STAGE);
  auto* red = reinterpret_cast<float*>(lds + NS * STAGE + V * RT * 8);
  const int lane = threadIdx.x % WAVE;
  if (__builtin_amdgcn_readfirstlane(threadIdx.x) >= NT) {
    const int tid = threadIdx.x - NT, wave = tid / WAVE;
    // Squares are added as rmsnorm_residual adds them, whose threads hold eight values side by
    // side: here two vectors of one thread, or those of two lanes, whose pairs are then of every
    // other thread there, so that two waves end where one wave's last step adds its halves.
    auto column = [&](int v) {
      if constexpr (V > 1) return (tid + v / 2 * RT) * 8 + v % 2 * 4;
      const int eight = wave / 2 * WAVE + (lane & ~1) + wave % 2;
      return eight * 8 + lane % 2 * 4;
    };
    floatx4 t[PARTS][V];
    u64b old[V], scale[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int c = min(column(v), K - 4);
#pragma unroll
      for (int p = 0; p < PARTS; ++p)
        t[p][v] = *reinterpret_cast<const floatx4*>(x + (long)min(p, S - 1) * K + c);
      old[v] = *reinterpret_cast<const u64b*>(res + c);
      scale[v] = *reinterpret_cast<const u64b*>(weight + c);
    }
    auto four = [](const unsigned short* v) {
      return (u64b)v[3] << 48 | (u64b)v[2] << 32 | (u64b)v[1] << 16 | v[0];
    };
    u64b kept[V];
    floatx4 y[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
      unsigned short b[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float sum = 0.f;
#pragma unroll
        for (int p = 0; p < PARTS; ++p) sum += p < S ? t[p][v][j] : 0.f;
        sum = bf16_to_f32(f32_to_bf16(sum)) + bf16_to_f32((unsigned short)(old[v] >> (16 * j)));
        b[j] = f32_to_bf16(sum);
        y[v][j] = column(v) < K ? sum : 0.f;
      }
      kept[v] = four(b);
    }
    auto squares = [&](const floatx4 a, float ss) {
#pragma unroll
      for (int j = 0; j < 4; ++j) ss = fmaf(a[j], a[j], ss);
      return ss;
    };
    if constexpr (V > 1) {
#pragma unroll
      for (int v = 0; v < V; v += 2) {
        const float ss = wave_sum(squares(y[v + 1], squares(y[v], 0.f)));
        if (lane == 0) red[v / 2 * (RT / WAVE) + wave] = ss;
      }
    } else {
      float ss = squares(y[0], __shfl_xor(squares(y[0], 0.f), 1, WAVE));  // odd lanes'
#pragma unroll
      for (int off = 32; off > 1; off >>= 1) ss += __shfl_xor(ss, off, WAVE);
      if (lane == 1) red[wave] = ss;
    }
    meet();
    float all = 0.f;
    if constexpr (V > 1) {
#pragma unroll
      for (int i = 0; i < V / 2 * (RT / WAVE); ++i) all += red[i];
    } else {
#pragma unroll
      for (int i = 0; i < RT / WAVE; i += 2) all += red[i] + red[i + 1];
    }
    const float inv = rsqrtf(all / K + eps);
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int c = column(v);
      unsigned short b[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        b[j] = f32_to_bf16(bf16_to_f32((unsigned short)(kept[v] >> (16 * j))) * inv *
                           bf16_to_f32((unsigned short)(scale[v] >> (16 * j))));
      *reinterpret_cast<u64b*>(row + c) = four(b);  // (past K: not read)
      if (blockIdx.x == 0 && blockIdx.y == 0 && c < K)
        *reinterpret_cast<u64b*>(res_out + c) = kept[v];
    }
    meet();
    return;  // barriers wait for the waves that are left
  }
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int at = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * (SILU ? WN / 2 : WN);
  const int k0 = blockIdx.y * span, steps = (min(K, k0 + span) - k0) / FEW_K;
  const unsigned short* src[L];
#pragma unroll
  for (int l = 0; l < L; ++l) {
    const int r = (tid + l * NT) >> 3, unit = (tid & 7) ^ (r & 7);
    const long n = SILU ? min(n0 + r / 16 * 8 + r % 8, N - 1) + (long)(r % 16 / 8) * N
                        : min(n0 + r, N - 1);
    src[l] = w + n * K + k0 + unit * 8;
  }
  auto issue = [&](int s) {
    char* stage = lds + s % NS * STAGE;
#pragma unroll
    for (int l = 0; l < L; ++l)
      __builtin_amdgcn_global_load_lds((gptr_t)(src[l] + (long)s * FEW_K),
                                       (lptr_t)(stage + (l * NT + wave * WAVE) * 16), 16, 0, 0);
  };
  for (int s = 0; s < min(steps, NS - 1); ++s) issue(s);
  meet();
  meet();
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  auto compute = [&](int s) {
    const char* stage = lds + s % NS * STAGE;
    frag_u wf[2], xf[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      wf[h].s = *reinterpret_cast<const shortx8*>(stage + (wave * 16 + at) * 128 +
                                                  ((h * 4 + g) ^ (at & 7)) * 16);
      xf[h].s = *reinterpret_cast<const shortx8*>(row + k0 + s * FEW_K + (h * 4 + g) * 8);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h].v, xf[h].v, acc, 0, 0, 0);
  };
  int s = 0;
  for (; s + NS - 1 < steps; ++s) {
    await_stage<(NS - 2) * L>();
    issue(s + NS - 1);  // over the stage before this, which all waves have left
    compute(s);
  }
  await_stage<0>();
  for (; s < steps; ++s) compute(s);
  if constexpr (SILU) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float up = __shfl_xor(acc[j], 32, WAVE);
      acc[j] = acc[j] / (1.f + __expf(-acc[j])) * up;
    }
    if (g >= 2) return;
  }
  if (at) return;  // all columns of the product are the row's
  const int n = n0 + (SILU ? wave * 8 + g * 4 : wave * 16 + g * 4);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (n + j < N) {
      if (!SILU && part) part[(long)blockIdx.y * N + n + j] = acc[j];
      else out[n + j] = f32_to_bf16(acc[j]);
    }
}

__global__ __launch_bounds__(256) void add_parts_kernel(const float* __restrict__ part,
                                                        unsigned short* __restrict__ out, int S,
                                                        long MN) {
  for (long i = blockIdx.x * 256L + threadIdx.x; i < MN; i += gridDim.x * 256L) {
    float sum = 0.f;
    for (int s = 0; s < S; ++s) sum += part[s * MN + i];
    out[i] = f32_to_bf16(sum);
  }
}

// [S, M, N] in fp32 -> their sum [M, N], rounded to bf16
torch::Tensor add_parts(const torch::Tensor& part) {
  const long S = part.size(0), M = part.size(1), N = part.size(2);
  auto out = torch::empty({M, N}, part.options().dtype(torch::kBFloat16));
  if (M * N == 0) return out;
  hipLaunchKernelGGL(add_parts_kernel, dim3(std::min((M * N + 255) / 256, 2048L)), dim3(256), 0,
                     CUR_STREAM, part.data_ptr<float>(), (unsigned short*)out.data_ptr(), (int)S,
                     M * N);
  HIP_CHECK_KERNEL();
  return out;
}

// K's parts: a workgroup per CU or a few less, of two stages at least (of weights that come
// from memory one CU takes in some 50 GB/s however much is under way, so more workgroups than
// CUs only even out badly; what lies in the L2 comes at 136 GB/s). 4096 x
// 14336, 23 rows: 1 part 52 us, 2 35, 4 23, 8 25; 2048 x 8192: 4 11.8, 8 9.3, 16 10.3; 4608
// x 3584: 2 11.1, 3 (216 workgroups) 9.3, 4 (288) 11.3.
static long parts_of(long N, long K) {
  const long tiles = std::max(1L, (N + 63) / 64);
  return std::max(1L, std::min({256 / tiles, K / FEW_K / 2, 16L}));
}

// Rows of W a workgroup takes and K's parts: what leaves a CU the least to read, of W at 21 GB/s
// when all read at once and of x at some 125, where the whole W does not take longer anyway
// (5.3 TB/s), and the reader the fewest parts; 64 rows unless 1.5 us are gained. Parts of a
// multiple of 2048 of K begin 4 KB apart, which tiles of more than 64 rows show (4608 x 14336, 8
// rows, 128 wide, 7 parts of 2048 35.7 us, 6 of 2432 29.2, 64 wide 27.9). Of 318 weights of 0.5 to
// 160 MB, 2 to 128 rows each, the norm that reads the parts included, the cut so chosen takes 1.4%
// longer than the best, 64 rows with the parts above 3.5%; one call in 90 is 3 to 8% behind the
// latter. us: 6144 x 4096, 1, 32, 64 and 96 rows, 64 wide 16.8 17.3 19.3 21.3, 96 wide in 4 parts
// 15.0 16.1 17.4 19.1; 8576 x 16064, 32 and 96 rows, 64 wide 73.7 100.4, 128 in 3 parts 56.2 66.9;
// 1536 x 1536, 8 parts, 64 and 128 rows 9.0 11.7, 96 wide in 12 10.0 13.4.
struct Cut {
  int width;
  long parts, rows = 0;
};
static Cut cut_of(long M, long N, long K) {
  const long steps = K / FEW_K, rows = M <= 32 ? 32 : (M + 31) / 32 * 32;
  Cut best = {64, 1};
  if (N == 0 || steps == 0) return best;
  // a single row's parts are read by a norm in the next product, which takes few (one_row_fits)
  if (M == 1 && N <= 4096) return {64, parts_of(N, K)};
  double low = 0;
  for (int width : {64, 96, 128}) {
    if (M == 1 && width > 96) break;  // (one_row_kernel has no wider form)
    const long tiles = (N + width - 1) / width;
    const long most = std::max(1L, std::min({256 / tiles, steps / 2, 16L}));
    for (long asked = most; asked >= std::max(1L, width > 64 ? most - 1 : most); --asked) {
      const long per = (steps + asked - 1) / asked, parts = (steps + per - 1) / per;
      const double cu = per * FEW_K * (width * 2 / 21. + rows * 2 * 0.4 / 50);
      double time = std::max(cu, N * K * 2 / 5300.) + parts * (M * N * 4 / 5000. + 50);
      if (width > 64) time = time * (parts > 1 && per % 32 == 0 ? 1.15 : 1) + 1500;
      if (low == 0 || time < low) low = time, best = {width, parts};
    }
  }
  return best;
}

static void check(const torch::Tensor& x, const torch::Tensor& w, long most = FEW_MOST) {
  TORCH_CHECK(x.is_cuda() && w.is_cuda() && x.dtype() == torch::kBFloat16 &&
                  w.dtype() == torch::kBFloat16 && w.is_contiguous(),
              "bf16 GPU only, contiguous weights");
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1) && x.size(0) <= most &&
                  x.size(1) % FEW_K == 0,
              "at most ", most, " rows and K a multiple of ", FEW_K);
}

// x as 16-byte loads can read its rows, which may be strided (a part of a joint projection,
// 64 rows of 256, copied first took 4.5 us more)
static torch::Tensor readable(const torch::Tensor& x) {
  const bool ok = x.dim() == 2 && (x.stride(1) == 1 || x.size(1) == 1) &&
                  (x.size(0) == 1 || (x.stride(0) >= x.size(1) && x.stride(0) % 8 == 0)) &&
                  (uintptr_t)x.data_ptr() % 16 == 0;
  // (contiguous() gives the same tensor back where only its address is odd)
  return ok ? x : x.clone(at::MemoryFormat::Contiguous);
}

template <int WN, int MT, bool SILU>
static void launch(const torch::Tensor& x, const torch::Tensor& w, unsigned short* out,
                   float* part, long N, long S, long span) {
  // stages: two workgroups of 64 rows on a CU, one of the wide forms
  constexpr int tile = SILU ? WN / 2 : WN, loads = (WN * 8 + MT * 128 + WN * 4 - 1) / (WN * 4);
  constexpr int NS = (WN == 64 ? 80 : 160) * 1024 / (loads * WN * 64);
  const long blocks = (x.size(0) + 16 * MT - 1) / (16 * MT);
  hipLaunchKernelGGL((few_rows_kernel<WN, MT, NS, SILU>), dim3((N + tile - 1) / tile, S, blocks),
                     dim3(WN * 4), 0, CUR_STREAM, (const unsigned short*)x.data_ptr(),
                     (const unsigned short*)w.data_ptr(), out, part, (int)x.size(0), (int)N,
                     (int)x.size(1), (int)span, x.size(0) > 1 ? x.stride(0) : 0L);
  HIP_CHECK_KERNEL();
}

// [M, N] in bf16, or with ``raw`` where K is cut [S, M, N] in fp32, S terms to be added.
static torch::Tensor cut_rows(torch::Tensor x, torch::Tensor w, bool raw, Cut cut,
                              long most = FEW_MOST) {
  check(x, w, most);
  x = readable(x);
  const long M = x.size(0), K = x.size(1), N = w.size(0);
  torch::Tensor out, part;
  if (M == 0 || N == 0 || K == 0) return torch::zeros({M, N}, x.options());
  const long steps = K / FEW_K;
  const long per = (steps + std::max(cut.parts, 1L) - 1) / std::max(cut.parts, 1L);
  const long S = (steps + per - 1) / per, span = per * FEW_K;
  if (S > 1) part = torch::empty({S, M, N}, x.options().dtype(torch::kFloat32));
  if (S == 1) out = torch::empty({M, N}, x.options());
  auto* op = S > 1 ? nullptr : (unsigned short*)out.data_ptr();
  float* pp = S > 1 ? part.data_ptr<float>() : nullptr;
  auto rows = [&](auto MT) {
    constexpr int mt = decltype(MT)::value;
    if (cut.width == 64) launch<64, mt, false>(x, w, op, pp, N, S, span);
    else if (cut.width == 96) launch<96, mt, false>(x, w, op, pp, N, S, span);
    else launch<128, mt, false>(x, w, op, pp, N, S, span);
  };
  const long high = cut.rows ? cut.rows : M;
  if (high <= 32) rows(std::integral_constant<int, 2>{});
  else if (high <= 64) rows(std::integral_constant<int, 4>{});
  else if (high <= 96) rows(std::integral_constant<int, 6>{});
  else rows(std::integral_constant<int, 8>{});
  if (S == 1) return out;
  return raw ? part : add_parts(part);
}

// The same in a given number of parts and rows of W a workgroup.
torch::Tensor few_rows(torch::Tensor x, torch::Tensor w, bool raw, long parts, long width,
                       long rows) {
  TORCH_CHECK(width == 64 || width == 96 || width == 128, "64, 96 or 128 rows of w a workgroup");
  return cut_rows(x, w, raw, Cut{(int)width, parts, rows}, rows ? 1 << 16 : FEW_MOST);
}

// How some hundred rows are cut: into blocks of ``rows``, each of which reads W once more, tiles
// of ``width`` and K's parts. A form's time is that of its stages of 64 of K, which depends on
// nothing but its rows and width while a CU has one workgroup (of 64 wide two share it), or what
// its XCDs read, if that takes longer: a tile's blocks lie on as many XCDs as their distance
// leaves over 8, and each of those reads the tile for itself (1408 x 8192, 400 rows, 64 x 128 in 3
// parts 35.7 us, 96 x 128 in 4, whose blocks share two, 25.1). Then there is what it takes to
// bring the parts to their reader. Fitted to 3516 sizes from 65 to 1000 rows and 512 x 576 to
// 8192 x 14336; the form so chosen takes 0.6% longer than the best measured.
static Cut block_cut(long M, long N, long K, bool raw) {
  static const struct {
    long rows;
    int width;
    float start, stage;  // us
  } forms[] = {{64, 64, 0.f, .27f}, {96, 64, .35f, .31f}, {64, 128, .7f, .365f},
               {96, 128, 1.2f, .453f}, {128, 128, 1.6f, .51f}};
  Cut best = {64, 1, 64};
  float low = 0;
  const long steps = K / FEW_K;
  for (const auto& f : forms) {
    const long across = (N + f.width - 1) / f.width, blocks = (M + f.rows - 1) / f.rows;
    const long most = std::max(1L, std::min({256 / (across * blocks), steps / 2, 16L}));
    for (long asked : {1L, most}) {
      const long per = (steps + asked - 1) / asked, parts = (steps + per - 1) / per;
      const long each = across * blocks * parts;
      const float full = each / 256.f;
      const float rounds = f.width > 64 ? (float)((each + 255) / 256)
                           : each <= 256 ? 1.f
                           : std::max(1.35f, full * (each <= 512 ? .92f : 1.15f));
      const long apart = across * parts % 8;  // blocks of a tile, in workgroups
      const long xcds = apart == 0 ? 1 : apart == 4 ? 2 : apart % 2 == 0 ? 4 : 8;
      const float way = N * K * 2e-6f / 7.f * std::min(blocks, xcds) +
                        M * K * 2e-6f / 12.f * std::min(across, 8L);
      const float time =
          f.start + std::max(per * f.stage * rounds, way) +
          (parts > 1 ? parts * M * N * (raw ? 1.55e-6f : 1.87e-6f) + (raw ? .4f : 3.f) : 0.f);
      if (low == 0 || time < low) low = time, best = {f.width, parts, f.rows};
    }
  }
  return best;
}

// How block_rows takes a product: 2 with K cut, 1 whole in one round of workgroups in which the
// blocks of a tile of W lie on one or two XCDs, else 0.
int block_form(long M, long N, long K, bool raw) {
  const Cut cut = block_cut(M, N, K, raw);
  if (cut.parts > 1) return 2;
  const long across = (N + cut.width - 1) / cut.width, blocks = (M + cut.rows - 1) / cut.rows;
  return across * blocks <= 256 && across % 4 == 0;
}

// linear_few_rows of more rows
torch::Tensor block_rows(torch::Tensor x, torch::Tensor w, bool raw) {
  return cut_rows(x, w, raw, block_cut(x.size(0), w.size(0), x.size(1), raw), 1 << 16);
}

// A router's logits in 16 parts [16, M, N] in fp32 that hold what the 16 waves of
// moe_route_kernel sum up, so that choices and weights do not depend on the number of tokens.
torch::Tensor router_rows(const torch::Tensor& x, const torch::Tensor& w) {
  check(x, w);
  const long M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(x.is_contiguous() && (uintptr_t)x.data_ptr() % 16 == 0 && M > 0 && N > 0,
              "contiguous tokens");
  auto part = torch::empty({16, M, N}, x.options().dtype(torch::kFloat32));
  // A wave takes 16 outputs of 16 rows (32 or 64 of 32 rows, in two or four waves: 64 x 2048, 64
  // tokens, 6.8 and 7.1 us, the choices included, and 6.5; 128 x 4096 10.4, 11.0 and 9.7).
  hipLaunchKernelGGL((few_rows_kernel<16, 1, 9, false, true>),
                     dim3((N + 15) / 16, 8, (M + 15) / 16), dim3(64), 0, CUR_STREAM,
                     (const unsigned short*)x.data_ptr(), (const unsigned short*)w.data_ptr(),
                     nullptr, part.data_ptr<float>(), (int)M, (int)N, (int)K, 0, K);
  HIP_CHECK_KERNEL();
  return part;
}

// ``steady``: as parts_of has K's parts, for any number of rows
torch::Tensor linear_few_rows(torch::Tensor x, torch::Tensor w, bool raw, bool steady) {
  // A kernel to add the parts pays off where a tile's steps take much longer than it: 2048
  // x 2048, 23 rows, 8.2 us whole, 4.0 and 4.7 in parts; 4096 x 4096 16.7, 8.9 and 2.4; 2048
  // x 2048, 64 rows, 11.7, 5.5 and 4.2.
  // More than 8192 outputs are cut for their reader alone: float_few_rows has their bits.
  const bool cut = raw || (x.size(1) * (x.size(0) > 32 ? 2 : 1) >= 4096 &&
                           parts_of(w.size(0), x.size(1)) > 1);
  const long M = x.size(0), N = w.size(0), K = x.size(1);
  return cut_rows(x, w, raw,
                  !cut ? Cut{64, 1} : steady ? Cut{64, parts_of(N, K)} : cut_of(M, N, K));
}

// linear_few_rows's result in float32, where K is not cut, without a kernel to convert it: 1 row
// of 32000 x 4096 59.8 and 57.1 us, 23 of 64128 x 2048 60.0 and 58.2, 64 of 32000 x 2048 37.9
// and 35.2.
bool float_few_rows_fits(long N, long K) { return parts_of(N, K) == 1; }
torch::Tensor float_few_rows(torch::Tensor x, torch::Tensor w) {
  check(x, w);
  x = readable(x);
  const long M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(M <= 64 && float_few_rows_fits(N, K), "at most 64 rows, K is cut for few outputs");
  auto out = torch::empty({M, N}, x.options().dtype(torch::kFloat32));
  if (M == 0 || N == 0) return out;
  float* pp = out.data_ptr<float>();
  auto* round = (unsigned short*)pp;
  if (M <= 32) launch<64, 2, false>(x, w, round, pp, N, 1, K);
  else launch<64, 4, false>(x, w, round, pp, N, 1, K);
  return out;
}

// silu(x @ gate^T) * (x @ up^T), rounded once; w: gate's rows, then up's
torch::Tensor silu_few_rows(torch::Tensor x, torch::Tensor w) {
  check(x, w);
  x = readable(x);
  TORCH_CHECK(w.size(0) % 2 == 0);
  const long M = x.size(0), K = x.size(1), N = w.size(0) / 2;
  auto out = torch::empty({M, N}, x.options());
  if (M == 0 || N == 0) return out;
  auto* op = (unsigned short*)out.data_ptr();
  // From 65 rows on x is as much to move as W: tiles of 128 halve it where there are enough
  // for the chip. 28672 x 4096, 96 rows, 59.9 and 56.1 us; 16384 x 2048 21.8 and 27.6; 28672
  // x 4096, 64 rows, 53.3 and 53.6. Tiles of 112 where one for every CU is enough: time with the
  // others over that with them, 33, 48, 64 and 96 rows:
  //   K      12288 outputs         13312                 14336
  //   1024   1.09 1.14 1.15 1.03   1.07 1.11 1.14 1.03   1.04 1.08 1.11 1.03
  //   2048   1.03 1.05 1.07 1.03   0.98 1.00 1.03 1.03   0.96 0.98 1.02 1.03
  //   3072   1.16 1.19 1.21 1.05   1.15 1.18 1.20 1.05   1.10 1.16 1.18 1.04
  //   3584   1.18 1.20 1.22 1.05   1.15 1.19 1.21 1.05   1.11 1.16 1.20 1.05
  //   4096   1.07 1.08 1.09 1.03   1.02 1.05 1.07 1.03   0.95 0.98 1.02 1.02
  // Rows of W 4 or 8 KB apart hold up tiles of 112 (28672 x 4096 4.6 TB/s, x 3584 5.5), so with
  // few rows of x and many outputs they stay at 64.
  const bool wide = N / 64 >= 192,
             one = wide && (N + 55) / 56 <= 256 && (M > 52 || K % 2048 || N <= 13056);
  auto rows = [&](auto MT) {
    constexpr int mt = decltype(MT)::value;
    if constexpr (mt > 2)
      if (one) return launch<112, mt, true>(x, w, op, nullptr, N, 1, K);
    if constexpr (mt > 4)
      if (wide) return launch<128, mt, true>(x, w, op, nullptr, N, 1, K);
    launch<64, mt, true>(x, w, op, nullptr, N, 1, K);
  };
  if (M <= 32) rows(std::integral_constant<int, 2>{});
  else if (M <= 64) rows(std::integral_constant<int, 4>{});
  else if (M <= 96) rows(std::integral_constant<int, 6>{});
  else rows(std::integral_constant<int, 8>{});
  return out;
}

// The kernel above where it has a form: x [S, 1, K] in fp32, S parts, of which a thread holds 64
// values at most. ``cut_of`` makes more for rows 1088 to 1792, 2112 to 3264 and 4160 to 6144
// wide, whose norms stay kernels of their own.
bool one_row_fits(long S, long K) {
  return S > 1 && K % FEW_K == 0 && K <= ROW_MOST &&
         S <= (K <= 1024 ? 16 : K <= 2048 ? 8 : K <= 4096 ? 4 : 2);
}

// w @ norm(x's parts + res), with ``silu`` as silu_few_rows, else as linear_few_rows's parts;
// the sum goes to res_out. ``steady``: K's parts as linear_few_rows then has them.
torch::Tensor one_row_product(torch::Tensor x, torch::Tensor res, torch::Tensor weight, double eps,
                              torch::Tensor res_out, torch::Tensor w, bool silu, bool steady) {
  TORCH_CHECK(x.is_cuda() && x.dtype() == torch::kFloat32 && x.is_contiguous() && x.dim() == 3 &&
                  x.size(1) == 1 && one_row_fits(x.size(0), x.size(2)),
              "a row in parts [S, 1, K]");
  const long S = x.size(0), K = x.size(2), N = silu ? w.size(0) / 2 : w.size(0);
  for (const auto& t : {res, weight, res_out, w})
    TORCH_CHECK(t.device() == x.device() && t.dtype() == torch::kBFloat16 && t.is_contiguous() &&
                    (uintptr_t)t.data_ptr() % 16 == 0, "bf16 beside the row, contiguous");
  TORCH_CHECK(res.numel() == K && weight.numel() == K && res_out.numel() == K &&
                  w.dim() == 2 && w.size(1) == K && w.size(0) % 2 == 0 && N > 0 &&
                  (uintptr_t)x.data_ptr() % 16 == 0 && res.data_ptr() != res_out.data_ptr(),
              "rows of K");
  const c10::DeviceGuard on(x.device());
  const Cut cut = silu ? Cut{64, 1} : steady ? Cut{64, parts_of(N, K)} : cut_of(1, N, K);
  const long steps = K / FEW_K, parts = cut.parts;
  const long per = (steps + parts - 1) / parts, S2 = (steps + per - 1) / per;
  torch::Tensor out, part;
  if (S2 > 1) part = torch::empty({S2, 1, N}, x.options());
  else out = torch::empty({1, N}, w.options());
  const int tile = silu ? 32 : cut.width;
  auto launch = [&](auto kern, int threads) {
    hipLaunchKernelGGL(kern, dim3((N + tile - 1) / tile, S2), dim3(threads), 0, CUR_STREAM,
                       x.data_ptr<float>(), (int)S, (const unsigned short*)res.data_ptr(),
                       (const unsigned short*)weight.data_ptr(),
                       (unsigned short*)res_out.data_ptr(), (float)eps,
                       (const unsigned short*)w.data_ptr(),
                       S2 > 1 ? nullptr : (unsigned short*)out.data_ptr(),
                       S2 > 1 ? part.data_ptr<float>() : nullptr, (int)N, (int)K,
                       (int)(per * FEW_K));
    HIP_CHECK_KERNEL();
  };
  auto form = [&](auto hv) {
    constexpr int HV = decltype(hv)::value;
    if (silu) launch(one_row_kernel<HV, true>, 256 + row_threads(HV));
    else if (cut.width == 64) launch(one_row_kernel<HV, false>, 256 + row_threads(HV));
    else launch(one_row_kernel<HV, false, 96>, 384 + row_threads(HV));
  };
  if (K <= 1024) form(std::integral_constant<int, 1>{});
  else if (K <= 2048) form(std::integral_constant<int, 2>{});
  else if (K <= 4096) form(std::integral_constant<int, 4>{});
  else form(std::integral_constant<int, 8>{});
  return S2 > 1 ? part : out;
}
