// Encoder-path kernels (gfx950): varlen self-attention without cache
// (bidirectional for the BGE-style embedder), mean-pool + L2 normalize.
//
// Replaces the reference's Weaviate text2vec-transformers sidecar
// (reference: docker-compose.yaml:545, routes/knowledge_base/weaviate_client.py:115)
// with on-GPU embedding.
#include "flash_tiles.h"
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

#define CUR_STREAM c10::hip::getCurrentHIPStream().stream()
#define ENC_KEYS 64   // keys per tile
#define ENC_ROWS 128  // query rows per workgroup
#define ENC_SLACK 10.f  // weights stay below 2^ENC_SLACK

// One head of 128 query rows per workgroup, 32 per wave, in the manner of the paged
// prompt kernel: S^T = K Q^T and O^T = V^T P^T, so a lane owns a row. Two tiles of 64 keys
// in LDS, the next one loaded while one is computed. Weights keep their 32 bits: each is
// the sum of three bf16 numbers (``split3``) and meets the values three times.
// Bound by memory and by the start of its many short sequences: 200 texts of 20 to 256
// tokens, 12 heads of 64 (170 MB) 676 us as a wave per row and head over scalar dot
// products, now 70 us.
// TURN: queries and keys are rotated here by their places in their sequence, a tile of keys
// in LDS as it arrives, and rounded as the rotation in memory rounds them (which reads and
// writes both: the same texts 27 us and 71 for the attention, together 82).
template <int D, bool TURN>
__global__ __launch_bounds__(256, 2) void packed_attn_kernel(
    const __hip_bfloat16* __restrict__ q,  // rows of Hq heads, D apart
    const __hip_bfloat16* __restrict__ k,  // rows of Hkv heads
    const __hip_bfloat16* __restrict__ v,
    __hip_bfloat16* __restrict__ out,  // [T, Hq, D]
    const int* __restrict__ cu, int S, int Hq, int Hkv, long qstride, long kstride,
    long vstride, float scale, int causal,
    const float* __restrict__ cos_sin, int places) {  // TURN: [places, D], cosines, then sines
  constexpr int NC = D / 16, NDT = D / 32, U = D / 8;
  constexpr int LU = ENC_KEYS * U / 256;  // loads per thread of K, and of V
  constexpr int KBYTES = ENC_KEYS * D * 2, STAGE = 2 * KBYTES;
  constexpr int KMASK = D == 128 ? 15 : 7;
  const int tid = threadIdx.x, lane = tid % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int col = lane & 31, half = lane >> 5;
  int seq, off;
  if (!find_block(cu, S, ENC_ROWS, blockIdx.x / Hq, lane, seq, off)) return;
  const int h = blockIdx.x % Hq, kvh = h / (Hq / Hkv);
  const long a = cu[seq];
  const int n = cu[seq + 1] - cu[seq];
  const int kend = causal ? min(n, off + ENC_ROWS) : n;
  const int ntiles = (kend + ENC_KEYS - 1) / ENC_KEYS;
  const int row0 = off + wave * 32, row = row0 + col;
  const bool valid = row < n;

  extern __shared__ __attribute__((aligned(16))) char smem[];
  const unsigned smem_at = (unsigned)(size_t)(__attribute__((address_space(3))) char*)smem;
  auto issue = [&](int tile) {
    char* st = smem + (tile & 1) * STAGE + wave * 64 * 16;
#pragma unroll
    for (int x = 0; x < LU; ++x) {
      const unsigned r = (tid + x * 256u) / U, slot = (tid + x * 256u) % U;
      const long t = a + min(tile * ENC_KEYS + (int)r, n - 1);  // past the end the last again
      const unsigned kd = (slot ^ (r & KMASK)) * 8;
      const unsigned vd = (slot ^ (D == 64 ? (r & 2) << 1 : (r & 3) << 2)) * 8;
      __builtin_amdgcn_global_load_lds((gptr_t)(k + t * kstride + kvh * D + kd),
                                       (lptr_t)(st + x * 256 * 16), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((gptr_t)(v + t * vstride + kvh * D + vd),
                                       (lptr_t)(st + KBYTES + x * 256 * 16), 16, 0, 0);
    }
  };
  issue(0);
  // of a token's rotation the cosines and sines of 8 pairs, from pair i on
  struct Angles {
    floatx4 c[2], s[2];
  };
  auto angles = [&](int t, int i) {
    const float* cs = cos_sin + (long)min(t, places - 1) * D + i;
    Angles y;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      y.c[k] = *reinterpret_cast<const floatx4*>(cs + 4 * k);
      y.s[k] = *reinterpret_cast<const floatx4*>(cs + D / 2 + 4 * k);
    }
    return y;
  };
  auto rotate = [](frag_u& u, frag_u& w, const Angles& y) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float a[2], b[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int e = 2 * j + k;
        const float c = y.c[e / 4][e % 4], s = y.s[e / 4][e % 4];
        const float x1 = __builtin_bit_cast(float, k ? u.u[j] & 0xffff0000u : u.u[j] << 16);
        const float x2 = __builtin_bit_cast(float, k ? w.u[j] & 0xffff0000u : w.u[j] << 16);
        a[k] = x1 * c - x2 * s;
        b[k] = x2 * c + x1 * s;
      }
      u.u[j] = cvt2_bf16(a[0], a[1]);
      w.u[j] = cvt2_bf16(b[0], b[1]);
    }
  };
  // a tile's rows have U / 2 pairs of units; a thread's
  constexpr int PAIRS = TURN ? ENC_KEYS * U / 2 / 256 : 1;
  Angles turn[PAIRS];
  auto prepare = [&](int tile) {
#pragma unroll
    for (int x = 0; x < PAIRS; ++x) {
      const int p = tid + x * 256;
      turn[x] = angles(min(tile * ENC_KEYS + p / (U / 2), n - 1), p % (U / 2) * 8);
    }
  };
  auto turn_keys = [&](int tile) {
#pragma unroll
    for (int x = 0; x < PAIRS; ++x) {
      const unsigned p = tid + x * 256u, r = p / (U / 2), unit = p % (U / 2);
      char* row = smem + (tile & 1) * STAGE + r * D * 2;
      shortx8* a = reinterpret_cast<shortx8*>(row + ((unit ^ (r & KMASK)) << 4));
      shortx8* b = reinterpret_cast<shortx8*>(row + (((unit + U / 2) ^ (r & KMASK)) << 4));
      frag_u u, w;
      u.s = *a;
      w.s = *b;
      rotate(u, w, turn[x]);
      *a = u.s;
      *b = w.s;
    }
  };
  if constexpr (TURN) prepare(0);

  // a scale that is not positive goes into the queries: the reference below compares
  // unscaled scores
  const unsigned flip = scale < 0.f ? 0x80008000u : 0u;
  const float c2 = scale == 0.f ? 1.f : fabsf(scale) * LOG2E;
  frag_u qf[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    qf[c].s = shortx8{0, 0, 0, 0, 0, 0, 0, 0};
    if (valid && scale != 0.f)
      qf[c].s = *reinterpret_cast<const shortx8*>(q + (a + row) * qstride + h * D + c * 16 +
                                                  half * 8);
  }
  if constexpr (TURN)
#pragma unroll
    for (int c = 0; c < NC / 2; ++c)
      rotate(qf[c], qf[c + NC / 2], angles(min(row, n - 1), c * 16 + half * 8));
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int j = 0; j < 4; ++j) qf[c].u[j] ^= flip;
  unsigned kat[NC], vat[NDT];
#pragma unroll
  for (int c = 0; c < NC; ++c)
    kat[c] = smem_at + col * D * 2 + (((c * 2 + half) ^ (col & KMASK)) << 4);
  {
    const int i = lane & 15, r = i >> 2, swz = D == 64 ? (r & 2) << 1 : r << 2;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
      const int unit = dt * 4 + ((lane >> 4) & 1) * 2 + ((i & 3) >> 1);
      vat[dt] = smem_at + KBYTES + (4 * half + r) * D * 2 + (unit ^ swz) * 16 + (i & 1) * 8;
    }
  }
  float m = -1e30f, l = 0.f;
  floatx16 o[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  const int wave_end = row0 >= n ? 0 : causal ? min(n, row0 + 32) : n;

  for (int tile = 0; tile < ntiles; ++tile) {
    // this tile is there for all, and nobody reads the other buffer any more
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if constexpr (TURN) turn_keys(tile);
    if (tile + 1 < ntiles) {
      issue(tile + 1);
      if constexpr (TURN) prepare(tile + 1);
    }
    if constexpr (TURN) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const unsigned st = (tile & 1) * STAGE;
    static_for<2>([&](auto SECOND) {
      constexpr int second = decltype(SECOND)::value;
      const int ks = tile * ENC_KEYS + second * 32;
      if (ks >= wave_end) return;
      floatx16 s;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        frag_u kf;
        kf.s = *(const __attribute__((address_space(3))) shortx8*)(kat[c] + st +
                                                                   second * 32 * D * 2);
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf.v, qf[c].v, s, 0, 0, 0);
      }
      const bool partly = ks + 31 >= n || (causal && ks + 31 > row0);
      if (partly) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = ks + (r & 3) + 8 * (r >> 2) + 4 * half;
          if (key >= n || (causal && key > row)) s[r] = -INFINITY;
        }
      }
      float mx = s[0];
#pragma unroll
      for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
      mx *= c2;
      if (__any(mx > m + ENC_SLACK)) {
        mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
        const float mn = fmaxf(m, mx), alpha = __builtin_amdgcn_exp2f(m - mn);
        m = mn;
        l *= alpha;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
      }
      frag_u pf[3][2];
      float sum = 0.f;
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        float p[2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
          p[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[2 * r + j], c2, -m));
        sum += p[0] + p[1];
        unsigned u[3];
        split3(p[0], p[1], u);
#pragma unroll
        for (int k = 0; k < 3; ++k) pf[k][r >> 2].u[r & 3] = u[k];
      }
      l += sum;
      // Where rows do not see all keys, infinite values stay out of the products, which
      // would make NaN of them and the others' 0, and are added to those who see them.
      const char* const vt = smem + st + KBYTES + second * 32 * D * 2;
      bool wild = false;
      if (partly) {
        unsigned most = 0;
#pragma unroll
        for (int x = 0; x < 32 * U / WAVE; ++x) {
          frag_u f;
          f.s = *reinterpret_cast<const shortx8*>(vt + (lane + x * WAVE) * 16);
#pragma unroll
          for (int j = 0; j < 4; ++j) most = max_halves(most, f.u[j] & 0x7fff7fffu);
        }
        wild = __any(most >= 0x7f800000u || (most & 0xffffu) >= 0x7f80u);
        if (wild)
          for (int t = 0; t < 32; ++t) {
            if (ks + t >= n || (causal && ks + t > row)) continue;
            const unsigned swz = D == 64 ? (t & 2) << 1 : (t & 3) << 2;
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
              for (int r = 0; r < 16; ++r) {
                const unsigned unit = dt * 4 + (r >> 2);
                const unsigned short y = *reinterpret_cast<const unsigned short*>(
                    vt + t * D * 2 + ((unit ^ swz) * 8 + 4 * half + (r & 3)) * 2);
                if ((y & 0x7f80u) == 0x7f80u) o[dt][r] += bf16_to_f32(y);
              }
          }
      }
      __builtin_amdgcn_sched_barrier(0);
      // pair i of V^T fragments: 16 keys i / (NDT / 2), d-tiles i % (NDT / 2) * 2 + {0, 1}
      shortx4 vf[NDT][4];
      auto fetch = [&](auto I) {
        constexpr int i = decltype(I)::value, ROW8 = 8 * D * 2;
        constexpr int at = second * 32 * D * 2 + i / (NDT / 2) * 2 * ROW8, dt = i % (NDT / 2) * 2;
        read_values<at, ROW8>(vf[i], vat[dt] + st, vat[dt + 1] + st);
      };
      fetch(std::integral_constant<int, 0>{});
      await_values(vf[0]);
      static_for<NDT>([&](auto I) {
        constexpr int i = decltype(I)::value, c = i / (NDT / 2), dt = i % (NDT / 2) * 2;
        if constexpr (i + 1 < NDT) fetch(std::integral_constant<int, i + 1>{});
        frag_u f[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          f[x].h[0] = vf[i][2 * x];
          f[x].h[1] = vf[i][2 * x + 1];
          if (wild)
#pragma unroll
            for (int j = 0; j < 4; ++j)
              f[x].u[j] &= ((f[x].u[j] & 0x7f80u) == 0x7f80u ? 0u : 0xffffu) |
                           ((f[x].u[j] & 0x7f800000u) == 0x7f800000u ? 0u : 0xffff0000u);
        }
#pragma unroll
        for (int k = 2; k >= 0; --k)
#pragma unroll
          for (int x = 0; x < 2; ++x)
            o[dt + x] =
                __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[x].v, pf[k][c].v, o[dt + x], 0, 0, 0);
        if constexpr (i + 1 < NDT) await_values(vf[i + 1]);
      });
    });
  }

  l += __shfl_xor(l, 32, WAVE);
  const float inv = 1.f / l;
  __hip_bfloat16* dst = out + ((a + row) * Hq + h) * D;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int g = 0; g < 4; g += 2) {
      unsigned y[2][2];
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          y[x][j] = cvt2_bf16(o[dt][4 * (g + x) + 2 * j] * inv,
                              o[dt][4 * (g + x) + 2 * j + 1] * inv);
      frag_u w;  // halves trade: 8 neighbouring channels of the row in one piece
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const auto r = __builtin_amdgcn_permlane32_swap(y[0][j], y[1][j], false, false);
        w.u[j] = r[0];
        w.u[2 + j] = r[1];
      }
      if (valid) *reinterpret_cast<shortx8*>(dst + dt * 32 + 8 * (g + half)) = w.s;
    }
}

// [T, H, D] whose rows may be strided, as 16-byte loads can read it
static torch::Tensor row_readable(const torch::Tensor& t) {
  const bool ok = t.stride(2) == 1 && (t.stride(1) == t.size(2) || t.size(1) == 1) &&
                  (t.stride(0) % 8 == 0 || t.size(0) == 1) &&
                  (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
  // (contiguous() gives the same tensor back where only its address is odd)
  return ok ? t : t.clone(at::MemoryFormat::Contiguous);
}

// ``cos_sin`` [places, D] fp32: queries and keys, not yet rotated, are turned by their places
// in their sequences, which must not be longer
static torch::Tensor packed_attention(const torch::Tensor& q_, const torch::Tensor& k_,
                                      const torch::Tensor& v_, const torch::Tensor& cu,
                                      double scale, bool causal,
                                      const c10::optional<torch::Tensor>& cos_sin) {
  TORCH_CHECK(q_.is_cuda() && q_.dtype() == torch::kBFloat16, "bf16 GPU only");
  const int T = q_.size(0), Hq = q_.size(1), D = q_.size(2), Hkv = k_.size(1);
  TORCH_CHECK(D == 64 || D == 128, "head_dim must be 64/128");
  TORCH_CHECK(k_.dtype() == q_.dtype() && v_.dtype() == q_.dtype() && k_.size(0) >= T &&
              v_.size(0) >= T && v_.size(1) == Hkv && k_.size(2) == D && v_.size(2) == D &&
              Hq % Hkv == 0 && cu.dtype() == torch::kInt32 && cu.is_contiguous(),
              "queries, keys and values");
  TORCH_CHECK(!cos_sin || (cos_sin->is_cuda() && cos_sin->dtype() == torch::kFloat32 &&
                           cos_sin->is_contiguous() && cos_sin->dim() == 2 &&
                           cos_sin->size(0) > 0 && cos_sin->size(1) == D &&
                           (reinterpret_cast<uintptr_t>(cos_sin->data_ptr()) & 15) == 0),
              "cosines and sines");
  auto out = torch::empty({T, Hq, D}, q_.options());
  const int S = cu.numel() - 1;
  if (T == 0 || S < 1) return out;
  const auto q = row_readable(q_), k = row_readable(k_), v = row_readable(v_);
  // as many blocks as there can be; each finds its rows, so that nothing is read back
  const dim3 grid((T / ENC_ROWS + S) * Hq), block(256);
  auto launch = [&](auto kern, int lds) {
    hipLaunchKernelGGL(kern, grid, block, lds, CUR_STREAM,
                       (const __hip_bfloat16*)q.data_ptr(), (const __hip_bfloat16*)k.data_ptr(),
                       (const __hip_bfloat16*)v.data_ptr(), (__hip_bfloat16*)out.data_ptr(),
                       cu.data_ptr<int>(), S, Hq, Hkv, q.stride(0), k.stride(0), v.stride(0),
                       (float)scale, causal ? 1 : 0,
                       cos_sin ? cos_sin->data_ptr<float>() : nullptr,
                       cos_sin ? (int)cos_sin->size(0) : 0);
  };
  if (D == 64 && cos_sin) launch(packed_attn_kernel<64, true>, 2 * 2 * ENC_KEYS * 64 * 2);
  else if (D == 64) launch(packed_attn_kernel<64, false>, 2 * 2 * ENC_KEYS * 64 * 2);
  else if (cos_sin) launch(packed_attn_kernel<128, true>, 2 * 2 * ENC_KEYS * 128 * 2);
  else launch(packed_attn_kernel<128, false>, 2 * 2 * ENC_KEYS * 128 * 2);
  HIP_CHECK_KERNEL();
  return out;
}

torch::Tensor attention_prefill(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                                torch::Tensor cu, double scale, bool causal) {
  return packed_attention(q, k, v, cu, scale, causal, c10::nullopt);
}

torch::Tensor attention_prefill_turned(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                                       torch::Tensor cos_sin, torch::Tensor cu, double scale,
                                       bool causal) {
  return packed_attention(q, k, v, cu, scale, causal, cos_sin);
}

// ---- mean-pool + L2 normalize per sequence -------------------------------

// A workgroup per sequence; H / 8 threads side by side take a row in 16-byte loads and
// 1024 / (H / 8) rows are under way at once (a thread per column and one row at a time
// before: 200 texts of 20 to 256 tokens of 768 236 us, now 12 us).
__global__ __launch_bounds__(1024) void embed_pool_kernel(
    const __hip_bfloat16* __restrict__ hidden, __hip_bfloat16* __restrict__ out,
    const int* __restrict__ cu, int H) {
  extern __shared__ float sums[];  // [row groups][H]
  __shared__ float s_norm[16];
  const int seq = blockIdx.x, a = cu[seq], b = cu[seq + 1];
  const int tid = threadIdx.x, nv = H / 8, groups = blockDim.x / nv;
  const int group = tid / nv, c = tid % nv * 8;
  if (group < groups) {
    float acc[8] = {};
#pragma unroll 4
    for (int t = a + group; t < b; t += groups) {
      const shortx8 x = *reinterpret_cast<const shortx8*>(hidden + (long)t * H + c);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] += bf16_to_f32((unsigned short)x[j]);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) sums[group * H + c + j] = acc[j];
  }
  __syncthreads();
  const float inv_n = 1.f / max(b - a, 1);
  float ss = 0.f;
  for (int d = tid; d < H; d += blockDim.x) {
    float y = 0.f;
    for (int g = 0; g < groups; ++g) y += sums[g * H + d];
    y *= inv_n;
    sums[d] = y;  // nobody else reads this column
    ss += y * y;
  }
  ss = wave_sum(ss);
  if (tid % WAVE == 0) s_norm[tid / WAVE] = ss;
  __syncthreads();
  float t = 0.f;
  for (int w = 0; w < (int)blockDim.x / WAVE; ++w) t += s_norm[w];
  const float inv = rsqrtf(t + 1e-24f);
  for (int d = tid; d < H; d += blockDim.x)
    *(unsigned short*)(out + (long)seq * H + d) = f32_to_bf16(sums[d] * inv);
}

// rows that are no multiple of 16 bytes: a thread per column
__global__ void embed_pool_any_kernel(const __hip_bfloat16* __restrict__ hidden,
                                      __hip_bfloat16* __restrict__ out,
                                      const int* __restrict__ cu, int H) {
  const int seq = blockIdx.x;
  const int a = cu[seq], b = cu[seq + 1];
  const int tid = threadIdx.x;
  __shared__ float s_norm[16];
  float acc[8];  // supports H <= 2048 at 256 threads
  const int nchunk = (H + blockDim.x - 1) / blockDim.x;
  for (int c = 0; c < nchunk; ++c) acc[c] = 0.f;
  for (int t = a; t < b; ++t)
    for (int c = 0; c < nchunk; ++c) {
      const int d = tid + c * blockDim.x;
      if (d < H)
        acc[c] += bf16_to_f32(*(const unsigned short*)(hidden + (long)t * H + d));
    }
  const float inv_n = 1.f / max(b - a, 1);
  float ss = 0.f;
  for (int c = 0; c < nchunk; ++c) {
    acc[c] *= inv_n;
    ss += acc[c] * acc[c];
  }
  ss = wave_sum(ss);
  if (tid % WAVE == 0) s_norm[tid / WAVE] = ss;
  __syncthreads();
  float t = 0.f;
  for (int w = 0; w < (int)blockDim.x / WAVE; ++w) t += s_norm[w];
  const float inv = rsqrtf(t + 1e-24f);
  for (int c = 0; c < nchunk; ++c) {
    const int d = tid + c * blockDim.x;
    if (d < H)
      *(unsigned short*)(out + (long)seq * H + d) = f32_to_bf16(acc[c] * inv);
  }
}

torch::Tensor embed_pool(torch::Tensor hidden, torch::Tensor cu) {
  TORCH_CHECK(hidden.is_cuda() && hidden.dtype() == torch::kBFloat16, "bf16 GPU only");
  const int H = hidden.size(1);
  TORCH_CHECK(H <= 2048, "embed_pool supports H <= 2048");
  const int S = cu.numel() - 1;
  auto out = torch::empty({S, H}, hidden.options());
  if (S == 0) return out;
  auto args = [&](auto kern, int threads, int lds) {
    hipLaunchKernelGGL(kern, dim3(S), dim3(threads), lds, CUR_STREAM,
                       (const __hip_bfloat16*)hidden.data_ptr(),
                       (__hip_bfloat16*)out.data_ptr(), cu.data_ptr<int>(), H);
  };
  if (H % 8 == 0 && (reinterpret_cast<uintptr_t>(hidden.data_ptr()) & 15) == 0)
    args(embed_pool_kernel, 1024, 1024 / (H / 8) * H * 4);
  else
    args(embed_pool_any_kernel, 256, 0);
  HIP_CHECK_KERNEL();
  return out;
}
