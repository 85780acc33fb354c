// Nearest documents of a few queries by inner product, for gfx950.
//
// Bound by one read of the documents. A wave scores 16 documents at a time for up to 16
// queries on the matrix cores: rows of the documents come straight as fragments, twelve
// loads of 1 KB in flight, queries from LDS. A workgroup keeps the scores of its documents
// in LDS as ordered integers and writes its best k; a second kernel merges those, so that
// scores never go through memory. Selection is by a bound: k lanes have a largest that
// reaches the k-th of all lanes' largest, so only what reaches it needs to be ranked.
// One query, 20 neighbours, 768 wide, before (a library product, its scores through memory
// and a library selection) and now: 1000000 documents in fp32 752 and 615 us (5.0 TB/s),
// in bf16 504 and 313; 100000 182 and 93, 102 and 58; 5000 52 and 25, 72 and 21. bf16 scores
// were rounded to bf16 before. What is left is the start and end of two kernels, some 20 us,
// and at a million the rate of a read.
#include "flash_tiles.h"
#include "plain.h"
#include <c10/core/DeviceGuard.h>
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

#define CUR_STREAM c10::hip::getCurrentHIPStream().stream()

#define KNN_WAVES 8
#define KNN_DOCS 1024     // most documents of a workgroup
#define KNN_QUERIES 16
#define KNN_MOST 64       // most neighbours
#define KNN_AHEAD 4       // groups of four loads: three under way, one in use
#define KNN_CHOSEN (2 * KNN_MOST + 32)  // most candidates of a wave
#define KNN_POOL 4096     // candidates that the merge ranks at a time

typedef unsigned long long key_t64;

// Order of floats as integers; NaN counts as the largest. 0 is below every float.
DEVINL unsigned ordered(float x) {
  const unsigned u = __builtin_bit_cast(unsigned, x);
  return x != x ? 0xffffffffu : u & 0x80000000u ? ~u : u | 0x80000000u;
}
DEVINL float unordered(unsigned u) {
  return __builtin_bit_cast(float, u == 0xffffffffu ? 0x7fc00000u
                                   : u & 0x80000000u ? u & 0x7fffffffu : ~u);
}

// The larger first, equal ones by place
DEVINL key_t64 join(unsigned value, unsigned place) {
  return (key_t64)value << 32 | (0xffffffffu - place);
}

DEVINL key_t64 shfl_xor64(key_t64 x, int d) {
  const unsigned lo = __shfl_xor((unsigned)x, d, WAVE);
  const unsigned hi = __shfl_xor((unsigned)(x >> 32), d, WAVE);
  return (key_t64)hi << 32 | lo;
}

// k-th largest of the lanes' keys
DEVINL key_t64 kth_of_wave(key_t64 x, int k, int lane) {
#pragma unroll
  for (int size = 2; size <= WAVE; size *= 2)
#pragma unroll
    for (int d = size / 2; d > 0; d /= 2) {
      const key_t64 y = shfl_xor64(x, d);
      const bool larger = ((lane & d) == 0) == ((lane & size) == 0);  // keeps the larger
      x = larger == (x > y) ? x : y;
    }
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)x, k - 1);
  const unsigned hi = __builtin_amdgcn_readlane((unsigned)(x >> 32), k - 1);
  return (key_t64)hi << 32 | lo;
}

// A bound that at least k of the wave's values reach and not many more: the k-th of the
// lanes' largest, raised by bisection while it lets through more than 2 k + 32. If that ends
// on equal values, ``above`` is the bound of the fewer than k larger ones, else the same.
DEVINL unsigned bound_of(const unsigned (&v)[KNN_DOCS / WAVE], int k, int lane,
                         unsigned& above) {
  unsigned best = 0;
#pragma unroll
  for (int i = 0; i < KNN_DOCS / WAVE; ++i) best = max(best, v[i]);
  unsigned lo = (unsigned)(kth_of_wave(join(best, lane), k, lane) >> 32), hi = 0xffffffffu;
  auto reached = [&](unsigned x) {
    int n = 0;
#pragma unroll
    for (int i = 0; i < KNN_DOCS / WAVE; ++i) n += __popcll(__ballot(v[i] >= x));
    return n;
  };
  above = lo;
  if (reached(lo) <= 2 * k + 32) return lo;
  if (reached(hi) >= k) return above = hi;  // as many NaN
  while (hi - lo > 1) {
    const unsigned mid = lo + (hi - lo) / 2;
    const int n = reached(mid);
    if (n < k) {
      hi = mid;
    } else {
      lo = mid;
      above = lo;
      if (n <= 2 * k + 32) return lo;
    }
  }
  above = hi;
  return lo;
}

// lists: [Q, workgroups, k] keys of the best of each workgroup's ``share`` documents
// (a multiple of 16), 0 where it has fewer than k. T: float or bf16 bits.
template <typename T>
__global__ __launch_bounds__(64 * KNN_WAVES, 4) void knn_score_kernel(
    const T* __restrict__ queries, const T* __restrict__ docs, key_t64* __restrict__ lists,
    long N, int D, int Q, int k, int share) {
  constexpr bool F32 = sizeof(T) == 4;
  constexpr int PER = 16 / sizeof(T);  // elements of a lane's load
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int row_bytes = D * (int)sizeof(T) + 16;  // 16 lanes' rows in different banks
  unsigned* scores = (unsigned*)(lds + Q * row_bytes);   // [Q][KNN_DOCS]
  key_t64* chosen = (key_t64*)(scores + Q * KNN_DOCS);  // [waves][KNN_CHOSEN]
  const int tid = threadIdx.x, lane = tid % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int at = lane & 15, g = lane >> 4;
  const long first = (long)blockIdx.x * share;
  const int count = (int)min((long)share, N - first);

  for (int x = tid; x < Q * D / PER; x += blockDim.x) {
    const int q = x / (D / PER), c = x % (D / PER);
    *(shortx8*)(lds + q * row_bytes + c * 16) = *(const shortx8*)(queries + (long)q * D + c * PER);
  }
  __syncthreads();

  // this wave's tiles of 16: wave, wave + 8, ..; groups of four steps of K through them
  const int tiles = (count + 15) / 16;
  const int groups = D / (16 * PER);
  const int mine = tiles > wave ? (tiles - wave + KNN_WAVES - 1) / KNN_WAVES : 0;
  const int total = mine * groups;
  frag_u buf[KNN_AHEAD][4];
  const char* src = nullptr;  // where the next group's rows are
  int tile = wave, left = 0;
  auto load = [&](auto B) {
    constexpr int b = decltype(B)::value;
    if (left == 0) {  // a lane's row of the next tile; past the end the last row again
      src = (const char*)(docs + (first + min(tile * 16 + at, count - 1)) * D) + g * 16;
      left = groups;
      if (tile + KNN_WAVES < tiles) tile += KNN_WAVES;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      buf[b][i].s = __builtin_nontemporal_load((const shortx8*)(src + i * 64));
    src += 256;
    --left;
  };
  floatx4 acc[4];
  int done = 0, group = 0;
  const char* qrow = lds + min(at, Q - 1) * row_bytes + g * 16;
  auto compute = [&](auto B) {
    constexpr int b = decltype(B)::value;
    if (group == 0)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      frag_u qf;
      qf.s = *(const shortx8*)(qrow + group * 256 + i * 64);
      if constexpr (F32) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
              __builtin_bit_cast(float, buf[b][i].u[j]), __builtin_bit_cast(float, qf.u[j]),
              acc[j], 0, 0, 0);
      } else {
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(buf[b][i].v, qf.v, acc[i], 0, 0, 0);
      }
    }
    if (++group == groups) {
      const floatx4 sum = (acc[0] + acc[1]) + (acc[2] + acc[3]);
      if (at < Q) {
        const int d0 = (wave + done * KNN_WAVES) * 16 + 4 * g;
#pragma unroll
        for (int r = 0; r < 4; ++r) scores[at * KNN_DOCS + d0 + r] = ordered(sum[r]);
      }
      group = 0;
      ++done;
    }
  };
  if (total > 0) {
    static_for<KNN_AHEAD>([&](auto b) { load(b); });
    for (int i = 0; i < total; i += KNN_AHEAD)
      static_for<KNN_AHEAD>([&](auto b) {
        if (i + b < total) compute(b);
        load(b);
        __builtin_amdgcn_sched_barrier(0);
      });
  }
  __syncthreads();

  // the best of the workgroup, a wave per query
  chosen += wave * KNN_CHOSEN;
  for (int q = wave; q < Q; q += KNN_WAVES) {
    unsigned v[KNN_DOCS / WAVE];
#pragma unroll
    for (int i = 0; i < KNN_DOCS / WAVE; ++i) {
      const int d = i * WAVE + lane;
      v[i] = d < count ? scores[q * KNN_DOCS + d] : 0;
    }
    unsigned above;
    const unsigned bound = max(bound_of(v, min(k, count), lane, above), 1u);
    int n = 0;
    auto take = [&](bool in, unsigned value, int d, int most) {
      const unsigned long long all = __ballot(in);
      const int to = n + __popcll(all & ((1ull << lane) - 1));
      if (in && to < most) chosen[to] = join(value, (unsigned)(first + d));
      n = min(n + __popcll(all), most);
    };
    above = max(above, 1u);
#pragma unroll
    for (int i = 0; i < KNN_DOCS / WAVE; ++i)
      take(v[i] >= above, v[i], i * WAVE + lane, KNN_CHOSEN);
    if (bound < above)  // equal ones in order until there are k
#pragma unroll
      for (int i = 0; i < KNN_DOCS / WAVE; ++i) take(v[i] == bound, v[i], i * WAVE + lane, k);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    key_t64* dst = lists + ((long)q * gridDim.x + blockIdx.x) * k;
    for (int i = lane; i < n; i += WAVE) {
      const key_t64 x = chosen[i];
      int rank = 0;
#pragma unroll 8
      for (int j = 0; j < n; ++j) rank += chosen[j] > x;
      if (rank < k) dst[rank] = x;
    }
    for (int i = n + lane; i < k; i += WAVE) dst[i] = 0;
    __builtin_amdgcn_wave_barrier();
  }
}

// A workgroup per query: the best k of ``count`` sorted lists of k. There are k in all.
__global__ __launch_bounds__(1024) void knn_merge_kernel(const key_t64* __restrict__ lists,
                                                         float* __restrict__ values,
                                                         long* __restrict__ indices, int count,
                                                         int k) {
  __shared__ key_t64 pool[KNN_POOL], bound_s;
  __shared__ unsigned tops[16][WAVE];
  __shared__ int held;
  const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
  const key_t64* mine = lists + (long)blockIdx.x * count * k;
  unsigned best = 0;
  // the lists' largest, and as many of the next as there are threads for
  const int depth = max(1, min(k, 1024 / count));
  for (int x = tid; x < count * depth; x += 1024)
    best = max(best, (unsigned)(mine[(long)(x % count) * k + x / count] >> 32));
  tops[wave][lane] = best;
  __syncthreads();
  if (wave == 0) {
    unsigned v[16], above;
#pragma unroll
    for (int w = 0; w < 16; ++w) v[w] = tops[w][lane];
    const unsigned b = bound_of(v, k, lane, above);
    if (lane == 0) bound_s = max((key_t64)b << 32, (key_t64)1);  // 0: fewer lists than k
  }
  for (;;) {
    if (tid == 0) held = 0;
    __syncthreads();
    const key_t64 bound = bound_s;
    for (int l = tid; l < count; l += 1024)
      for (int i = 0; i < k; ++i) {
        const key_t64 x = mine[(long)l * k + i];
        if (x < bound) break;
        const int to = atomicAdd(&held, 1);
        if (to < KNN_POOL) pool[to] = x;
      }
    __syncthreads();
    const int all = held, n = min(all, KNN_POOL);
    for (int i = tid; i < n; i += 1024) {
      const key_t64 x = pool[i];
      int rank = 0;
#pragma unroll 8
      for (int j = 0; j < n; ++j) rank += pool[j] > x;
      if (all > KNN_POOL) {  // a higher bound that k of the pool reach; far fewer are left
        if (rank == k - 1) bound_s = x;
      } else if (rank < k) {
        values[(long)blockIdx.x * k + rank] = unordered((unsigned)(x >> 32));
        indices[(long)blockIdx.x * k + rank] = 0xffffffffu - (unsigned)x;
      }
    }
    if (all <= KNN_POOL) return;
    __syncthreads();
  }
}

template <typename T>
static std::vector<torch::Tensor> nearest(const torch::Tensor& query, const torch::Tensor& docs,
                                          int k) {
  const long Q = query.size(0), D = query.size(1), N = docs.size(0);
  const c10::DeviceGuard on(docs.device());
  // about two workgroups per CU, which hold 1024 at most: 400000 documents, 768 floats, 256
  // 298 us, 512 264, 1024 306
  const long share = std::min<long>(KNN_DOCS, std::max<long>(128, (N / 512 + 127) / 128 * 128));
  const long blocks = (N + share - 1) / share;
  auto lists = torch::empty({Q, blocks, k}, query.options().dtype(torch::kInt64));
  auto values = torch::empty({Q, k}, query.options().dtype(torch::kFloat32));
  auto indices = torch::empty({Q, k}, query.options().dtype(torch::kInt64));
  const int lds = Q * (D * sizeof(T) + 16) + Q * KNN_DOCS * 4 + KNN_WAVES * KNN_CHOSEN * 8;
  auto kern = knn_score_kernel<T>;
  static const hipError_t once = hipFuncSetAttribute(
      (const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  (void)once;
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(64 * KNN_WAVES), lds, CUR_STREAM,
                     (const T*)query.data_ptr(), (const T*)docs.data_ptr(),
                     (key_t64*)lists.data_ptr(), N, (int)D, (int)Q, k, (int)share);
  hipLaunchKernelGGL(knn_merge_kernel, dim3(Q), dim3(1024), 0, CUR_STREAM,
                     (const key_t64*)lists.data_ptr(), values.data_ptr<float>(),
                     indices.data_ptr<long>(), (int)blocks, k);
  HIP_CHECK_KERNEL();
  return {values, indices};
}

std::vector<torch::Tensor> knn_topk(torch::Tensor query, torch::Tensor docs, long k) {
  TORCH_CHECK(query.is_cuda(), "GPU only");
  query = query.to(docs.dtype());
  k = std::min<long>(k, docs.size(0));
  const long size = docs.element_size();
  const bool f32 = docs.dtype() == torch::kFloat32;
  // Rows in whole groups of four 64-byte steps, as many queries as a fragment has columns
  // and as many neighbours as a wave has lanes. Within
  // that the kernels won at every size tried, most narrowly with 3 queries and 1 neighbour:
  // 607 and 667 us at a million in fp32, 27 and 31 at 5000; 16 queries and 40 neighbours 649
  // and 852. The library's product serves the rest, and all that autograd, a transform or a
  // trace follows.
  if (plain(query) && plain(docs) && docs.is_cuda() && query.dim() == 2 && docs.dim() == 2 && query.size(1) == docs.size(1) &&
      (f32 || docs.dtype() == torch::kBFloat16) && docs.is_contiguous() &&
      query.is_contiguous() && query.size(1) > 0 && query.size(1) * size % 256 == 0 &&
      query.size(1) * size <= 4096 && query.size(0) > 0 && query.size(0) <= KNN_QUERIES &&
      k > 0 && k <= KNN_MOST && docs.size(0) < 0xffffffffL &&
      (uintptr_t)docs.data_ptr() % 16 == 0 && (uintptr_t)query.data_ptr() % 16 == 0 &&
      docs.device() == query.device())
    return f32 ? nearest<float>(query, docs, (int)k) : nearest<unsigned short>(query, docs, (int)k);
  auto scores = torch::mm(query, docs.t()).to(torch::kFloat32);
  auto [vals, idx] = scores.topk(k, -1);
  return {vals, idx};
}
