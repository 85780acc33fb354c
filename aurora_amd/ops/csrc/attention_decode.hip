// Paged-KV decode attention for gfx950 (one new token per sequence).
//
// Memory-bound by the KV read; a workgroup streams a stretch of one (sequence, kv head)
// once for up to 16 query heads of the group, four waves taking 32 keys in turn:
//  * scores are S^T = K Q^T and results O^T = V^T P^T on the matrix cores, so a lane owns
//    a head and maxima, sums and rescaling need no exchange. Keys come from the cache
//    straight as A fragments; values through registers and the wave's own LDS, from where
//    transposing reads give V^T with its keys in the order in which the scores lie. Nothing
//    is shared between waves until the end, so there is no barrier in the loop;
//  * the next 32 keys and values are under way while 32 are computed (16 KB a wave);
//  * weights keep their 32 bits: each is the sum of three bf16 numbers (``split3``) and
//    meets the values three times; O is rescaled only when a score exceeds the reference by DEC_SLACK powers
//    of two;
//  * contexts are cut into stretches of equal length, found on the device from all context
//    lengths (``split_length``), so that a few long ones do not keep the others waiting
//    and few sequences still fill the chip; the last workgroup to end merges the stretches
//    of a sequence that has several.
// Measured in a graph, before and now (a second kernel that merges, whole contexts in the order of
// the batch): 96 sequences of 500 to 2900 keys, 32 heads over 8, 128 wide, 143 and 124 us (5.4
// TB/s; a large read reaches 5.5 to 5.8), the same in fp8 86 and 82; 256 of 1600 292 (5.8 TB/s);
// one of 12000 29.5 and 19.0, one of 777 13.3 and 10.2, 8 of 200 to 600 15.8 and 12.2; 7 heads
// over one, 4 fp8 sequences of 3000 to 9000 27.7 and 18.8; fp8 64 wide, 23 of 300 to 5000, 27.6
// and 24.4. A single sequence is bound by trips to memory one behind the other: lengths, pages,
// keys, and to merge a mark and the other stretches.
//
// Replaces the per-token provider round-trip of the reference agent loop
// (reference: server/chat/backend/agent/llm.py:192) with an in-process
// batched decode step.
#include "flash_tiles.h"
#include "head_turn.h"
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

#define CUR_STREAM c10::hip::getCurrentHIPStream().stream()

#define DEC_KEYS 32       // keys a wave takes at a time
#define DEC_WAVES 4
#define DEC_HEADS 16      // query heads of a workgroup
#define DEC_SLACK 10.f    // weights stay below 2^DEC_SLACK
#define DEC_TARGET 1024   // stretches that the contexts are cut into
#define DEC_LEAST 160     // of few keys each

enum { FROM_WHOLE = 1, FROM_PARTS = 2 };  // what a kernel that rotates finds
enum { NO_BIAS = 0, LINEAR_BIAS = 1, LOG_BIAS = 2, FLAT_BIAS = 3 };

// keys of a sequence that its query sees: [first, L)
struct Seen {
  int window, chunk;
  DEVINL int first(int L) const {
    int lo = window > 0 ? max(0, L - window) : 0;
    if (chunk > 0 && L > 0) lo = max(lo, L - 1 - (L - 1) % chunk);
    return lo;
  }
};

// Keys per stretch, a multiple of 128 (one round of the waves): what leaves about DEC_TARGET
// stretches over all sequences and head tiles; of less than 512 only to have DEC_LEAST of them, as
// a stretch takes its start and many take longer to merge than they save. 8 kv heads, us with
// stretches of at least 128, 256, 384 and 512: one sequence of 777 keys 10.1 11.0 12.0 13.0, of
// 4000 16.1 13.2 14.0 13.9, of 12000 33 23 20 19; 8 of 300 to 1500 15.7 16.5 14.2 14.9; 16 of 1024
// 28 21 23 21; 16 of 100 to 3000 34 34 34 30. All lanes of a wave.
DEVINL int split_length(const int* ctx, int B, int tiles, const Seen& seen, int lane) {
  long sum = 0;
  for (int s = lane; s < B; s += WAVE) sum += ctx[s] - seen.first(ctx[s]);
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) sum += __shfl_xor(sum, d, WAVE);
  const long per = (sum * tiles + DEC_TARGET - 1) / DEC_TARGET;
  const long least = min(max(sum * tiles / DEC_LEAST, 1L), 512L);
  return (int)((max(per, least) + 127) / 128 * 128);
}

DEVINL int splits_of(int seen, int length) { return max(1, (seen + length - 1) / length); }

// sequence and place of stretch ``idx``, the sequence's first stretch and their number
DEVINL bool find_split(const int* ctx, int B, int length, const Seen& seen, int idx, int lane,
                       int& b, int& s, int& n) {
  for (int b0 = 0; b0 < B; b0 += WAVE) {
    const int x = b0 + lane;
    const int c = x < B ? splits_of(ctx[x] - seen.first(ctx[x]), length) : 0;
    int end = c;
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
      const int before = __shfl_up(end, d, WAVE);
      if (lane >= d) end += before;
    }
    const unsigned long long past = __ballot(end > idx);
    if (past) {
      const int at = __builtin_ctzll(past);
      b = b0 + at;
      n = __builtin_amdgcn_readlane(c, at);
      s = idx - (__builtin_amdgcn_readlane(end, at) - n);
      return true;
    }
    idx -= __builtin_amdgcn_readlane(end, WAVE - 1);
  }
  return false;
}

// Workgroups that each take a whole context start by length, longest first: the last to start
// are short. (32 heads over 8, 128 wide, in the order of the batch and so: 96 sequences of 500 to
// 2900 keys 143 and 124 us, all of their mean 119; 128 of 50 to 1500 87 and 80; 64 of 300 to 8000
// 232 and 220; 41 of 700 to 2600 74 and 66; 100 of 600 56.2 and 57.1, of 50 16.2 and 16.6.) The
// sequence whose context is the idx-th longest, to between a 64th and a 32nd of the
// longest, in the batch's order where they are alike, and its length; of at most 64 N. All
// lanes of a wave.
template <int N>
DEVINL int ranked(const int* ctx, int B, int idx, int lane, int& length) {
  int n[N], most = 0;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const int s = lane + k * WAVE;
    n[k] = s < B ? ctx[s] : 0;
    most = max(most, n[k]);
  }
  auto take = [&](int at) {
#pragma unroll
    for (int k = 0; k < N; ++k)
      if (at >> 6 == k) length = __builtin_amdgcn_readlane(n[k], at & 63);
    return at;
  };
  idx = __builtin_amdgcn_readfirstlane(idx);
  if (!__any(most > 512)) return take(idx);  // an order costs half a microsecond
  // the highest bit of any
  int bits = 0;
#pragma unroll
  for (int step = 16; step > 0; step >>= 1)
    if (__any(most >> (bits + step) != 0)) bits += step;
  const int shift = max(bits - 5, 0);
  unsigned long long in[N];
  bool less = false, two = false, three = false;  // quarters of that bit's double
#pragma unroll
  for (int k = 0; k < N; ++k) {
    in[k] = __ballot(lane + k * WAVE < B);
    const int v = n[k] >> (shift + 4);
    if (lane + k * WAVE < B) less |= v < 2, two |= v == 2, three |= v == 3;
  }
  if (!__any(less) && !(__any(two) && __any(three))) return take(idx);  // alike
#pragma unroll
  for (int bit = 5; bit >= 0; --bit) {
    unsigned long long one[N];
    int count = 0;
#pragma unroll
    for (int k = 0; k < N; ++k) {
      one[k] = __ballot(n[k] >> (shift + bit) & 1) & in[k];
      count += __popcll(one[k]);
    }
    const bool here = idx < count;
    if (!here) idx -= count;
#pragma unroll
    for (int k = 0; k < N; ++k) in[k] = here ? one[k] : in[k] & ~one[k];
  }
  int at = 0;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const int c = __popcll(in[k]);
    if (idx >= 0 && idx < c) {
      const unsigned long long below = (1ull << lane) - 1;
      const bool is = (in[k] >> lane & 1) && __popcll(in[k] & below) == idx;
      at = k * WAVE + __builtin_ctzll(__ballot(is));
    }
    idx -= c;
  }
  return take(__builtin_amdgcn_readfirstlane(at));
}

// Four V^T fragments at once: rows 4 g .. and 16 + 4 g .. of d-tiles at four addresses.
template <int SECOND>
DEVINL void read_value_tiles(shortx4 (&v)[8], unsigned a0, unsigned a1, unsigned a2,
                             unsigned a3) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n\t"
      "ds_read_b64_tr_b16 %1, %8 offset:%12\n\t"
      "ds_read_b64_tr_b16 %2, %9\n\t"
      "ds_read_b64_tr_b16 %3, %9 offset:%12\n\t"
      "ds_read_b64_tr_b16 %4, %10\n\t"
      "ds_read_b64_tr_b16 %5, %10 offset:%12\n\t"
      "ds_read_b64_tr_b16 %6, %11\n\t"
      "ds_read_b64_tr_b16 %7, %11 offset:%12\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]),
        "=&v"(v[6]), "=&v"(v[7])
      : "v"(a0), "v"(a1), "v"(a2), "v"(a3), "n"(SECOND)
      : "memory");
}

// Numbers that workgroups on different XCDs hand each other go past the L2s, each of which
// knows only its own: made known by a fence instead, every workgroup would write its whole L2
// back and drop it (23 sequences of 300 to 5000 keys 27 and 60 us).
DEVINL void hand_over(float* p, float x) {
  __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
DEVINL float handed(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Results of two heads, h by half a wave, from the n stretches of their sequence, ``src`` the
// first one's. 32 references and sums are read at once, and the first results with them.
template <int DV, bool TURNS>
DEVINL void merge_stretches(const float* src, long step, int n, int lane, __hip_bfloat16* out,
                            int b, int h, int L, long ostride, int dv, float oscale,
                            const float* sink, const HeadTurn& turn) {
  constexpr int N = DV / 32, AT_ONCE = 8;
  const int col = lane & 31;
  float M = sink ? fmaxf(sink[h] * LOG2E, -1e30f) : -1e30f, Lsum = sink ? 1.f : 0.f, O[N] = {};
  for (int s0 = 0; s0 < n; s0 += 32) {
    float o[AT_ONCE][N];
    auto read = [&](int first) {
#pragma unroll
      for (int k = 0; k < AT_ONCE; ++k)
#pragma unroll
        for (int j = 0; j < N; ++j)
          o[k][j] = handed(src + min(first + k, n - 1) * step + col + j * 32);
    };
    const float* ref = src + min(s0 + col, n - 1) * step + DV;
    const float m = s0 + col < n ? handed(ref) : -1e30f, l = s0 + col < n ? handed(ref + 1) : 0.f;
    read(s0);
    float most = m;
#pragma unroll
    for (int d = 16; d > 0; d >>= 1) most = fmaxf(most, __shfl_xor(most, d, WAVE));
    const float Mn = fmaxf(M, most), alpha = __builtin_amdgcn_exp2f(M - Mn);
    M = Mn;
    const float f = s0 + col < n ? __builtin_amdgcn_exp2f(m - M) : 0.f;
    float sum = f * l;
#pragma unroll
    for (int d = 16; d > 0; d >>= 1) sum += __shfl_xor(sum, d, WAVE);
    Lsum = Lsum * alpha + sum;
#pragma unroll
    for (int j = 0; j < N; ++j) O[j] *= alpha;
    for (int s = s0; s < min(s0 + 32, n); s += AT_ONCE) {
      if (s > s0) read(s);
#pragma unroll
      for (int k = 0; k < AT_ONCE; ++k) {
        const float fk = __shfl(f, (lane & 32) + (s - s0 + k), WAVE);
#pragma unroll
        for (int j = 0; j < N; ++j)
          if (s + k < n) O[j] += fk * o[k][j];
      }
    }
  }
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int d = col + j * 32;
    float y = O[j] / Lsum * oscale;
    if constexpr (TURNS) y = turned<bf16_t>(turn, y, b, L - 1, h, d, dv);
    if (d < dv) *(unsigned short*)(out + b * ostride + (long)h * dv + d) = f32_to_bf16(y);
  }
}

// What a step's projection left of its queries and of the new keys and values: rows [B, width] of
// queries, keys and values side by side, in bf16 or in ``parts`` fp32 terms ``step`` apart, to
// which a bias is added, and the rotations [positions, D]. A row is the last of its sequence.
struct Fresh {
  const void* qkv;
  const unsigned short* bias;
  const float* cos_sin;
  void *kc, *vc;
  int parts;
  long step;
  bool by_eight;  // the order of sums of the separate kernel's form of many rows
};

bool rotates_by_eight(long T, long width);  // defined in elementwise.hip

// BIAS: a distance penalty per head or none (see attention_prefill.hip), a window or
// chunks of positions; sink: one more term of the denominator per head, or null;
// FLAT_BIAS results may be turned back and gated. PAGED: pages are whole tiles.
// Without CUT a workgroup takes a whole context.
// FRESH: the workgroup adds up and rotates its queries itself, and that of the last stretch the
// new key and value, which it writes to the cache and takes from LDS where the cache would still
// have what was there before. While parts and rotations are on their way so are its first keys.
// After a kernel of its own for that and with it in here, 32 heads over 8, us: one sequence of
// 777, 128 wide, 12.0 and 10.1; 8 of 300 to 1500 17.2 and 14.7; 41 of 700 to 2600 71.0 and 68.7;
// 23 of 300 to 5000 in fp8 48.3 and 45.5, 64 wide 27.1 and 25.0. Where whole contexts fill the chip
// the work takes as long here (96 of 500 to 2900 124.5 and 4.8, in one 129.2) and what goes is the
// launch between: captured steps of 8 layers 4096 wide 2316 and 2302, 64 sequences 1998 and
// 1957, 128 of 300 to 1500 2247 and 2230, in fp8 1950 and 1901.
// (Four columns and partners a lane in all waves, with 64-bit addresses, gave half of that.)
template <int D, int DV, bool FP8, int BIAS, bool PAGED, bool CUT, int FRESH = 0>
__global__ __launch_bounds__(256, FRESH && D == 64 ? 4 : 2) void paged_decode_kernel(
    const __hip_bfloat16* __restrict__ q,   // [B, Hq, D]
    // (not __restrict__: loads of them must stay before the waits that count them)
    const void* kc,  // [NP, Hkv, P, D] bf16 | fp8 e4m3
    const void* vc,
    __hip_bfloat16* out,                    // [B, ostride], heads dv apart
    float* part,                            // [stretches, Hq, DV + 2], where a context has several
    int* arrived,                           // [B, head tiles] zeros, and again at the end
    const int* __restrict__ block_tables,   // [B, MP]
    const int* __restrict__ ctx_lens,       // [B]
    int B, int Hq, int Hkv, int P, int MP, float scale,
    long ostride, int dv, float oscale,
    const float* __restrict__ slopes, const float* __restrict__ rates, Seen seen,
    const float* __restrict__ sink, HeadTurn turn, Fresh fresh) {
  static_assert(!FRESH || (PAGED && !BIAS && D == DV));
  constexpr int NC = D / 32, NDT = DV / 16;
  constexpr int EB = FP8 ? 1 : 2;
  constexpr int VU = DV / 8, LV = DEC_KEYS * VU / WAVE;  // 16-B units of a value, a lane's
  constexpr int STAGE = DEC_KEYS * DV * 2;
  const int lane = threadIdx.x % WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int G = Hq / Hkv, NG = (G + DEC_HEADS - 1) / DEC_HEADS;
  const int tiles = Hkv * NG, idx = blockIdx.x / tiles, tile = blockIdx.x % tiles;
  const int kvh = tile / NG, h0 = kvh * G + tile % NG * DEC_HEADS;
  const int GT = min(DEC_HEADS, kvh * G + G - h0);
  int b = idx, split = 0, nsplits = 1, length = 0x7fffffff, L = -1;
  // LDS: a tile of values per wave; at the end the waves' results
  __shared__ __attribute__((aligned(16))) char smem[DEC_WAVES * STAGE];
  __shared__ float s_m[DEC_WAVES][DEC_HEADS], s_l[DEC_WAVES][DEC_HEADS];
  static_assert(sizeof(smem) >= DEC_WAVES * DEC_HEADS * DV * 4);
  if (!CUT && seen.window <= 0 && seen.chunk <= 0) {
    if (B <= 2 * WAVE) b = ranked<2>(ctx_lens, B, idx, lane, L);
    else if (B <= 4 * WAVE) b = ranked<4>(ctx_lens, B, idx, lane, L);
  }
  if (CUT) {
    length = split_length(ctx_lens, B, tiles, seen, lane);
    if (!find_split(ctx_lens, B, length, seen, idx, lane, b, split, nsplits)) return;
    // the same in all lanes, which the compiler cannot see
    b = __builtin_amdgcn_readfirstlane(b);
    split = __builtin_amdgcn_readfirstlane(split);
    nsplits = __builtin_amdgcn_readfirstlane(nsplits);
    length = __builtin_amdgcn_readfirstlane(length);
  }
  if (L < 0) L = ctx_lens[b];
  const int first = seen.first(L);
  const int t_lo = first + (CUT ? split * length : 0);
  const int t_hi = CUT ? min(L, t_lo + length) : L;
  const int* bt = block_tables + (long)b * MP;
  const int head = lane & 15, g = lane >> 4;
  const bool mine = head < GT;

  char* ring = smem + wave * STAGE;
  const unsigned ring_at =
      (unsigned)(size_t)(__attribute__((address_space(3))) char*)ring;

  frag_u qf[NC];
  if constexpr (!FRESH) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      qf[c].s = shortx8{0, 0, 0, 0, 0, 0, 0, 0};
      if (mine)
        qf[c].s = *reinterpret_cast<const shortx8*>(q + ((long)b * Hq + h0 + head) * D + c * 32 +
                                                    g * 8);
    }
  }
  const float c2 = scale * LOG2E;  // scores in units of log 2
  const float slope = BIAS == LINEAR_BIAS && mine ? slopes[h0 + head] * LOG2E
                      : BIAS == LOG_BIAS && mine  ? slopes[h0 + head] : 0.f;
  const float rate = BIAS == LOG_BIAS && mine ? rates[h0 + head] : 0.f;

  float m = -1e30f, l = 0.f;
  floatx4 o[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) o[dt] = floatx4{0.f, 0.f, 0.f, 0.f};

  // this wave's tiles: t0 + 128 i. Row of key t in a head's cache; past the end the last
  // key again
  const int t_end = FRESH ? max(t_hi, 1) : t_hi;
  auto row_of = [&](int t) -> long {
    t = min(t, t_end - 1);
    return ((long)bt[t / P] * Hkv + kvh) * P + t % P;
  };
  auto value_unit = [&](int x, int& row, int& col) {
    const unsigned u = lane + x * WAVE;
    row = u / VU;
    col = ((u % VU) ^ (DV == 64 ? (row >> 1 & 3) << 1 : (row & 7) << 1)) * 8;
  };
  // (Through registers and not straight to LDS: beside direct-to-LDS loads the compiler
  // turns every wait for a register into a wait for all loads.)
  using raw = std::conditional_t<FP8, u64b, shortx8>;
  raw kr[2][2][NC], vr[LV];   // K: [parity][16 keys][32 dimensions]
  // Rows of a tile: past the end the last tile again, so that every round has as many
  // loads. PAGED: its first row is looked up a tile ahead.
  long page_row = 0;
  auto tile_at = [&](int t0) { return min(t0, (t_end - 1) & -DEC_KEYS); };
  auto lookup = [&](int t0) {
    if constexpr (PAGED) page_row = row_of(tile_at(t0));
  };
  auto source = [&](int t0, int key, long first_row) -> long {
    t0 = tile_at(t0);
    // (the table need not name pages behind a window)
    if constexpr (!PAGED) return row_of(BIAS ? max(t0 + key, t_lo) : t0 + key);
    return first_row + (t0 + DEC_KEYS <= t_end ? key : min(key, t_end - 1 - t0));
  };
  auto load_keys = [&](int t0, long first_row, auto PARITY) {
    constexpr int parity = decltype(PARITY)::value;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const char* src = (const char*)kc + (source(t0, k * 16 + head, first_row) * D + g * 8) * EB;
#pragma unroll
      for (int c = 0; c < NC; ++c)
        kr[parity][k][c] = *reinterpret_cast<const raw*>(src + c * 32 * EB);
    }
  };
  auto load_values = [&](int t0, long first_row) {
#pragma unroll
    for (int x = 0; x < LV; ++x) {
      int row, col;
      value_unit(x, row, col);
      vr[x] = *reinterpret_cast<const raw*>(
          (const char*)vc + (source(t0, row, first_row) * DV + col) * EB);
    }
  };
  auto widen = [](raw x) -> shortx8 {
    if constexpr (FP8) return fp8x8_to_bf16x8(x);
    else return x;
  };
  // where a lane's values lie: lane i of 16 reads 8 bytes of row 4 g + i / 4
  const int vrow = 4 * g + (head >> 2);
  const unsigned vat = ring_at + vrow * DV * 2, vcol =
      ((((head & 3) >> 1) ^ (DV == 64 ? (vrow >> 1 & 3) << 1 : (vrow & 7) << 1)) << 4) +
      (head & 1) * 8;

  // FRESH: queries as bf16, the new key and value as the cache has them
  __shared__ __attribute__((aligned(16))) unsigned short s_q[FRESH ? DEC_HEADS * D : 8];
  __shared__ __attribute__((aligned(16))) char s_kv[FRESH ? 2 * D * EB : 16];
  const bool ends = FRESH && t_hi == L;  // this stretch is the last

  // one round: the tile at t0, whose keys are in kr[parity] and whose values in vr; the
  // wave's next tile is requested as soon as its registers are free
  constexpr int ROUND = DEC_WAVES * DEC_KEYS;
  auto compute = [&](int t0, auto PARITY) {
    constexpr int parity = decltype(PARITY)::value;
    const long next_row = page_row;
    load_keys(t0 + ROUND, next_row, std::integral_constant<int, 1 - parity>{});
    lookup(t0 + 2 * ROUND);
    __builtin_amdgcn_sched_barrier(0);
    const bool newest = ends && t0 + DEC_KEYS >= L;
    if (FRESH && newest) {
      int own = lane;
      asm volatile("" : "+v"(own));  // nothing of this is kept through the rounds
#pragma unroll
      for (int k = 0; k < 2; ++k)
        if (t0 + k * 16 + (own & 15) == L - 1)
#pragma unroll
          for (int c = 0; c < NC; ++c)
            kr[parity][k][c] =
                *reinterpret_cast<const raw*>(s_kv + (c * 32 + (own >> 4) * 8) * EB);
    }
    floatx4 st[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      st[k] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        frag_u kf;
        kf.s = widen(kr[parity][k][c]);
        st[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf.v, qf[c].v, st[k], 0, 0, 0);
      }
    }
    float x[8];  // scores of keys 16 k + 4 g + r
    float mx = -INFINITY;
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = t0 + k * 16 + 4 * g + r;
        float y = st[k][r] * c2;
        if constexpr (BIAS == LINEAR_BIAS || BIAS == LOG_BIAS) {
          const float dist = (float)(L - 1 - t);
          y -= slope * (BIAS == LOG_BIAS ? __builtin_amdgcn_logf(1.f + rate * dist) : dist);
        }
        if (t >= t_hi || (BIAS && t < t_lo)) y = -INFINITY;
        x[k * 4 + r] = y;
        mx = fmaxf(mx, y);
      }
    if (__any(mx > m + DEC_SLACK)) {
      mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE));
      mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
      const float mn = fmaxf(m, mx), alpha = __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) o[dt] *= alpha;
    }
    frag_u pf[3];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float p0 = __builtin_amdgcn_exp2f(x[2 * j] - m);
      const float p1 = __builtin_amdgcn_exp2f(x[2 * j + 1] - m);
      l += p0 + p1;
      unsigned u[3];
      split3(p0, p1, u);
#pragma unroll
      for (int k = 0; k < 3; ++k) pf[k].u[j] = u[k];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < LV; ++x)
      *reinterpret_cast<shortx8*>(ring + (lane + x * WAVE) * 16) = widen(vr[x]);
    if (t0 + DEC_KEYS > t_hi || (BIAS && t0 < t_lo)) {
      // keys that nobody sees: what stands in their place may be infinite
#pragma unroll
      for (int x = 0; x < LV; ++x) {
        const int t = t0 + (lane + x * WAVE) / VU;
        if (t >= t_hi || (BIAS && t < t_lo))
          *reinterpret_cast<shortx8*>(ring + (lane + x * WAVE) * 16) =
              shortx8{0, 0, 0, 0, 0, 0, 0, 0};
      }
    }
    if (FRESH && newest) {
      int own = lane;
      asm volatile("" : "+v"(own));  // the same
      const int row = L - 1 - t0;  // its units lie side by side
      if (own < VU) {
        const int turn = DV == 64 ? (row >> 1 & 3) << 1 : (row & 7) << 1;
        *reinterpret_cast<shortx8*>(ring + (row * VU + own) * 16) =
            widen(*reinterpret_cast<const raw*>(s_kv + (D + (own ^ turn) * 8) * EB));
      }
    }
    load_values(t0 + ROUND, next_row);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d4 = 0; d4 < NDT; d4 += 4) {
      shortx4 v[8];
      read_value_tiles<16 * DV * 2>(v, vat + (vcol ^ (d4 * 32)), vat + (vcol ^ (d4 * 32 + 32)),
                                    vat + (vcol ^ (d4 * 32 + 64)), vat + (vcol ^ (d4 * 32 + 96)));
#pragma unroll
      for (int k = 2; k >= 0; --k)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          frag_u vf;
          vf.h[0] = v[2 * j];
          vf.h[1] = v[2 * j + 1];
          o[d4 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, pf[k].v, o[d4 + j], 0, 0, 0);
        }
    }
  };
  using EVEN = std::integral_constant<int, 0>;
  using ODD = std::integral_constant<int, 1>;
  // tiles lie within pages, so the first may begin before the stretch
  int t0 = t_lo - (BIAS ? t_lo % DEC_KEYS : 0) + wave * DEC_KEYS;
  if constexpr (FRESH) {
    // Two columns of a head and their partners half a head on, of all that is new, a lane; waves
    // that find nothing left ask for their keys alone. (All of a wave's work here stands in the way
    // of the others on its SIMD: offsets are 32 bits beside addresses that all lanes share.)
    constexpr int UNITS = D / 4, HALF = D / 2, AHEAD = 8;
    const int all = (GT + 2 * ends) * UNITS;
    lookup(t0);
    auto request = [&] {  // (waves without a tile ask for the last one too: a branch here
                          // would make the others wait for all their loads)
      load_keys(t0, page_row, EVEN{});
      load_values(t0, page_row);
    };
    const long row = (long)b * (Hq + 2 * Hkv) * D;
    const float* turns = fresh.cos_sin + (long)max(L - 1, 0) * D;
    const bool keep = ends && L > 0 && tile % NG == 0;
    long slot = 0;
    if (keep) slot = (((long)bt[(L - 1) / P] * Hkv + kvh) * P + (L - 1) % P) * D;
    auto take = [&](int x, auto meanwhile) {
      const unsigned h = (unsigned)x / UNITS, i = (unsigned)x % UNITS * 2;
      const bool is_q = h < (unsigned)GT, is_v = h > (unsigned)GT;  // queries, the key, the value
      const unsigned column = (is_q ? h0 + h : is_v ? Hq + Hkv + kvh : Hq + kvh) * D + i;
      floatx2 part[AHEAD][2], y[2];
      unsigned whole[2], bias[2] = {0, 0};
      if constexpr (FRESH == FROM_PARTS) {
#pragma unroll
        for (int p = 0; p < AHEAD; ++p) {
          const float* src = (const float*)fresh.qkv + row + min(p, fresh.parts - 1) * fresh.step;
#pragma unroll
          for (int z = 0; z < 2; ++z)
            part[p][z] = *reinterpret_cast<const floatx2*>(src + (column + z * HALF));
        }
      } else {
        const auto* src = (const bf16_t*)fresh.qkv + row;
#pragma unroll
        for (int z = 0; z < 2; ++z)
          whole[z] = *reinterpret_cast<const unsigned*>(src + (column + z * HALF));
      }
      const floatx2 cs = *reinterpret_cast<const floatx2*>(turns + i),
                    sn = *reinterpret_cast<const floatx2*>(turns + (i + HALF));
      if (fresh.bias)
#pragma unroll
        for (int z = 0; z < 2; ++z)
          bias[z] = *reinterpret_cast<const unsigned*>(fresh.bias + (column + z * HALF));
      meanwhile();
      __builtin_amdgcn_sched_barrier(0);
      auto round = [](floatx2 v) {
        const unsigned u = cvt2_bf16(v[0], v[1]);
        return floatx2{__uint_as_float(u << 16), __uint_as_float(u & 0xffff0000u)};
      };
      auto two = [](unsigned u) {
        return floatx2{__uint_as_float(u << 16), __uint_as_float(u & 0xffff0000u)};
      };
#pragma unroll
      for (int z = 0; z < 2; ++z)
        if constexpr (FRESH == FROM_PARTS) {
          y[z] = floatx2{0.f, 0.f};
#pragma unroll
          for (int p = 0; p < AHEAD; ++p)
            if (p < fresh.parts) y[z] += part[p][z];
        } else {
          y[z] = two(whole[z]);
        }
      if constexpr (FRESH == FROM_PARTS) {
        for (int p = AHEAD; p < fresh.parts; ++p)
#pragma unroll
          for (int z = 0; z < 2; ++z)
            y[z] += *reinterpret_cast<const floatx2*>((const float*)fresh.qkv + row +
                                                      p * fresh.step + (column + z * HALF));
        y[0] = round(y[0]), y[1] = round(y[1]);
      }
      if (fresh.bias) y[0] = round(y[0] + two(bias[0])), y[1] = round(y[1] + two(bias[1]));
      if (!is_v)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const float x1 = y[0][j], x2 = y[1][j];
          y[0][j] = __builtin_fmaf(x1, cs[j], -(x2 * sn[j]));
          y[1][j] = fresh.by_eight ? __builtin_fmaf(x1, sn[j], x2 * cs[j])
                                   : __builtin_fmaf(x2, cs[j], x1 * sn[j]);
        }
      if (is_q) {
#pragma unroll
        for (int z = 0; z < 2; ++z)
          *reinterpret_cast<unsigned*>(s_q + h * D + i + z * HALF) = cvt2_bf16(y[z][0], y[z][1]);
        return;
      }
      using pair = std::conditional_t<FP8, unsigned short, unsigned>;
      char* cache = (char*)(is_v ? fresh.vc : fresh.kc) + (slot + i) * EB;
#pragma unroll
      for (int z = 0; z < 2; ++z) {
        pair v;
        if constexpr (FP8) v = (pair)__builtin_amdgcn_cvt_pk_fp8_f32(y[z][0], y[z][1], 0u, false);
        else v = cvt2_bf16(y[z][0], y[z][1]);
        *reinterpret_cast<pair*>(s_kv + ((is_v ? D : 0) + i + z * HALF) * EB) = v;
        if (keep) *reinterpret_cast<pair*>(cache + z * HALF * EB) = v;
      }
    };
    if (wave * WAVE < all) take(min((int)threadIdx.x, all - 1), request);
    else request();
    for (int x0 = DEC_WAVES * WAVE; x0 + wave * WAVE < all; x0 += DEC_WAVES * WAVE)
      take(min(x0 + (int)threadIdx.x, all - 1), [] {});
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (keys stay on their way)
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      qf[c].s = shortx8{0, 0, 0, 0, 0, 0, 0, 0};
      if (mine) qf[c].s = *reinterpret_cast<const shortx8*>(s_q + head * D + c * 32 + g * 8);
    }
  }
  if (t0 < t_hi) {
    if constexpr (!FRESH) {
      lookup(t0);
      load_keys(t0, page_row, EVEN{});
      load_values(t0, page_row);
    }
    lookup(t0 + ROUND);
    for (;;) {
      compute(t0, EVEN{});
      if ((t0 += ROUND) >= t_hi) break;
      compute(t0, ODD{});
      if ((t0 += ROUND) >= t_hi) break;
    }
  }

  // ---- the waves' results
  l += __shfl_xor(l, 16, WAVE);
  l += __shfl_xor(l, 32, WAVE);
  __syncthreads();
  float* so = (float*)smem;  // [waves][heads][DV]
  if (mine) {
    if (g == 0) {
      s_m[wave][head] = m;
      s_l[wave][head] = l;
    }
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
      *reinterpret_cast<floatx4*>(so + (wave * DEC_HEADS + head) * DV + dt * 16 + 4 * g) = o[dt];
  }
  __syncthreads();
  for (int gd = threadIdx.x; gd < GT * DV; gd += blockDim.x) {
    const int hh = gd / DV, d = gd % DV;
    const bool ends = BIAS && nsplits == 1 && sink;  // the sink counts once
    const float s0 = ends ? fmaxf(sink[h0 + hh] * LOG2E, -1e30f) : -1e30f;
    float M = s0;
#pragma unroll
    for (int w = 0; w < DEC_WAVES; ++w) M = fmaxf(M, s_m[w][hh]);
    float Lsum = ends ? __builtin_amdgcn_exp2f(s0 - M) : 0.f, O = 0.f;
#pragma unroll
    for (int w = 0; w < DEC_WAVES; ++w) {
      const float f = __builtin_amdgcn_exp2f(s_m[w][hh] - M);
      Lsum += f * s_l[w][hh];
      O += f * so[(w * DEC_HEADS + hh) * DV + d];
    }
    if (nsplits == 1) {
      float y = O / Lsum * oscale;
      if constexpr (BIAS == FLAT_BIAS) y = turned<bf16_t>(turn, y, b, L - 1, h0 + hh, d, dv);
      if (!BIAS || d < dv)
        *(unsigned short*)(out + b * ostride + (long)(h0 + hh) * dv + d) = f32_to_bf16(y);
    } else {
      // an un-normalised partial result, its reference and its sum
      float* dst = part + ((long)idx * Hq + h0 + hh) * (DV + 2);
      hand_over(dst + d, O);
      if (d == 0) {
        hand_over(dst + DV, M);
        hand_over(dst + DV + 1, Lsum);
      }
    }
  }
  if (nsplits == 1) return;
  // The last workgroup of the sequence's head tile to come here merges its stretches: all
  // waves' results have left the CU before one thread makes them known and learns of others'.
  __shared__ int s_last;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    int* mark = arrived + (long)b * tiles + tile;
    const int before =
        __hip_atomic_fetch_add(mark, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = before == nsplits - 1;
    if (s_last) *mark = 0;
  }
  __syncthreads();
  if (!s_last) return;
  for (int hh = 2 * wave + lane / 32; hh < GT; hh += 2 * DEC_WAVES)
    merge_stretches<DV, BIAS == FLAT_BIAS>(part + ((long)(idx - split) * Hq + h0 + hh) * (DV + 2),
                                           (long)Hq * (DV + 2), nsplits, lane, out, b, h0 + hh, L,
                                           ostride, dv, oscale, BIAS ? sink : nullptr, turn);
}

// Marks that a call wants for its sequences' head tiles, or 0 where contexts stay whole: while
// the longest that can be seen is short or the workgroups are many, cutting costs its search
// and the merge, and evens out little. Whole and cut, 128 wide, 8 kv heads: 32 sequences of 1024
// keys 31 and 34 us, 96 of 100 to 3000 115 and 132, 16 of 1024 21 and 21; on the other side
// 4 sequences of 3000 to 9000 keys 93 and 30, 23 of 300 to 5000 73 and 61, 32 of 300 to 8000 126
// and 114. What it gives up: 64 sequences of 300 to 8000 keys 221 and 215.
long decode_marks(long B, long Hq, long Hkv, long longest, long window, long chunk) {
  const long tiles = Hkv * ((Hq / Hkv + DEC_HEADS - 1) / DEC_HEADS);
  if (window > 0) longest = std::min(longest, window);
  if (chunk > 0) longest = std::min(longest, chunk);
  return longest > std::max<long>(256, B * tiles * B * tiles / 16) ? B * tiles : 0;
}

template <int D, int DV, bool FP8, int BIAS, int FRESH = 0>
static void decode_launch(const torch::Tensor& q, const torch::Tensor& kc,
                          const torch::Tensor& vc, const torch::Tensor& bt,
                          const torch::Tensor& ctx, __hip_bfloat16* out, long ostride,
                          int dv, float scale, float oscale, const float* slopes,
                          const float* rates, int window, int chunk, const float* sink,
                          const HeadTurn& turn,
                          const c10::optional<torch::Tensor>& marks, const Fresh& fresh = {}) {
  const int B = q.size(0), Hq = q.size(1);
  const int Hkv = kc.size(1), P = kc.size(2), MP = bt.size(1);
  const int tiles = Hkv * ((Hq / Hkv + DEC_HEADS - 1) / DEC_HEADS);
  const bool cut = decode_marks(B, Hq, Hkv, (long)MP * P, window, chunk) > 0;
  const long most = cut ? B + DEC_TARGET / tiles + 1 : B;  // stretches there can be
  torch::Tensor part, arrived;
  if (cut) {
    part = torch::empty({most, Hq, DV + 2}, q.options().dtype(torch::kFloat32));
    const bool fit = marks && marks->dtype() == torch::kInt32 && marks->device() == q.device() &&
                     marks->is_contiguous() && marks->numel() >= (long)B * tiles;
    arrived = fit ? *marks : torch::zeros({(long)B * tiles}, ctx.options());
  }
  float* pp = cut ? part.data_ptr<float>() : nullptr;
  const Seen seen = {window, chunk};
  auto launch = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(most * tiles), dim3(256), 0, CUR_STREAM,
                       (const __hip_bfloat16*)q.data_ptr(), kc.data_ptr(), vc.data_ptr(), out,
                       pp, cut ? arrived.data_ptr<int>() : nullptr, bt.data_ptr<int>(),
                       ctx.data_ptr<int>(), B, Hq, Hkv, P, MP,
                       scale, ostride, dv, oscale, slopes, rates, seen, sink, turn, fresh);
  };
  const bool paged = P % DEC_KEYS == 0;
  if constexpr (FRESH) {
    if (cut) launch(paged_decode_kernel<D, DV, FP8, BIAS, true, true, FRESH>);
    else launch(paged_decode_kernel<D, DV, FP8, BIAS, true, false, FRESH>);
  } else if (paged && cut) launch(paged_decode_kernel<D, DV, FP8, BIAS, true, true>);
  else if (paged) launch(paged_decode_kernel<D, DV, FP8, BIAS, true, false>);
  else if (cut) launch(paged_decode_kernel<D, DV, FP8, BIAS, false, true>);
  else launch(paged_decode_kernel<D, DV, FP8, BIAS, false, false>);
  HIP_CHECK_KERNEL();
}

torch::Tensor paged_attention_decode(torch::Tensor q, torch::Tensor kc,
                                     torch::Tensor vc, torch::Tensor bt,
                                     torch::Tensor ctx, double scale,
                                     c10::optional<torch::Tensor> into,
                                     c10::optional<torch::Tensor> marks) {
  TORCH_CHECK(q.is_cuda() && q.dtype() == torch::kBFloat16, "bf16 GPU only");
  const int B = q.size(0), Hq = q.size(1), D = q.size(2), Hkv = kc.size(1);
  TORCH_CHECK(Hq % Hkv == 0, "GQA requires Hq % Hkv == 0");
  TORCH_CHECK(D == 128 || D == 64, "unsupported head_dim ", D);
  auto out = result_like(q, into);
  if (B == 0) return out;
  auto* o = (__hip_bfloat16*)out.data_ptr();
  const long stride = (long)Hq * D;
  const bool fp8 = kc.dtype() == torch::kFloat8_e4m3fn;
#define RUN(DD, F8) \
  decode_launch<DD, DD, F8, NO_BIAS>(q, kc, vc, bt, ctx, o, stride, D, (float)scale, \
                                     1.f, nullptr, nullptr, 0, 0, nullptr, HeadTurn{}, marks)
  if (D == 128) { if (fp8) RUN(128, true); else RUN(128, false); }
  else { if (fp8) RUN(64, true); else RUN(64, false); }
#undef RUN
  return out;
}

// The same of rows that are the last of their sequences, none of which comes twice: ``qkv`` [B,
// (Hq + 2 Hkv) D] is the projection, whole or in parts, to which a bias is added; the new keys and
// values go where the tables have the last of ``ctx`` positions. Nothing where there is no form.
c10::optional<torch::Tensor> fresh_attention_decode(
    torch::Tensor qkv, c10::optional<torch::Tensor> bias, torch::Tensor cos_sin, torch::Tensor kc,
    torch::Tensor vc, torch::Tensor bt, torch::Tensor ctx, long Hq, double scale,
    c10::optional<torch::Tensor> marks) {
  const bool raw = qkv.dtype() == torch::kFloat32 && qkv.dim() == 3;
  if (!qkv.is_cuda() || !qkv.is_contiguous() || (!raw && qkv.dtype() != torch::kBFloat16))
    return {};
  const long B = qkv.size(raw ? 1 : 0), Hkv = kc.size(1), P = kc.size(2), D = kc.size(3);
  const long width = (Hq + 2 * Hkv) * D;
  const bool fp8 = kc.dtype() == torch::kFloat8_e4m3fn;
  if (B == 0 || (D != 64 && D != 128) || vc.size(3) != D || Hq % Hkv || P % DEC_KEYS ||
      qkv.dim() != (raw ? 3 : 2) || qkv.size(-1) != width || vc.dtype() != kc.dtype() ||
      (!fp8 && kc.dtype() != torch::kBFloat16) || cos_sin.dtype() != torch::kFloat32 ||
      cos_sin.dim() != 2 || cos_sin.size(1) != D || bt.dim() != 2 || bt.size(0) != B ||
      ctx.numel() != B ||
      bt.dtype() != torch::kInt32 || ctx.dtype() != torch::kInt32 ||
      (bias && (bias->dtype() != torch::kBFloat16 || bias->numel() != width)))
    return {};
  for (const torch::Tensor* t : {&qkv, &kc, &vc, &cos_sin, bias ? &*bias : &qkv, &bt, &ctx})
    if (t->device() != qkv.device() || !t->is_contiguous() ||
        (t != &bt && t != &ctx && (uintptr_t)t->data_ptr() % 16))
      return {};
  auto out = torch::empty({B, Hq, D}, qkv.options().dtype(torch::kBFloat16));
  const Fresh fresh = {qkv.data_ptr(), bias ? (const unsigned short*)bias->data_ptr() : nullptr,
                       cos_sin.data_ptr<float>(), kc.data_ptr(), vc.data_ptr(),
                       raw ? (int)qkv.size(0) : 1, B * width, rotates_by_eight(B, width)};
#define RUN1(DD, F8, HOW)                                                                   \
  decode_launch<DD, DD, F8, NO_BIAS, HOW>(out, kc, vc, bt, ctx, o, Hq* D, DD, (float)scale, \
                                          1.f, nullptr, nullptr, 0, 0, nullptr, HeadTurn{}, \
                                          marks, fresh)
#define RUN(DD, F8) if (raw) RUN1(DD, F8, FROM_PARTS); else RUN1(DD, F8, FROM_WHOLE)
  auto* o = (__hip_bfloat16*)out.data_ptr();
  if (D == 128) { if (fp8) { RUN(128, true); } else { RUN(128, false); } }
  else { if (fp8) { RUN(64, true); } else { RUN(64, false); } }
#undef RUN
#undef RUN1
  return out;
}

void biased_attention_decode(torch::Tensor q, torch::Tensor kc, torch::Tensor vc,
                             torch::Tensor bt, torch::Tensor ctx, double scale,
                             long window, long chunk, c10::optional<torch::Tensor> slopes,
                             c10::optional<torch::Tensor> rates,
                             c10::optional<torch::Tensor> sink,
                             c10::optional<torch::Tensor> turn,
                             c10::optional<torch::Tensor> gate, torch::Tensor out,
                             long col, long dv, double oscale,
                             c10::optional<torch::Tensor> marks) {
  TORCH_CHECK(q.is_cuda() && q.dtype() == torch::kBFloat16 && q.is_contiguous());
  const int B = q.size(0), Hq = q.size(1), D = q.size(2);
  const int Hkv = kc.size(1), DV = vc.size(3);
  TORCH_CHECK(Hq % Hkv == 0 && kc.size(3) == D && vc.size(1) == Hkv &&
              vc.size(2) == kc.size(2));
  TORCH_CHECK(kc.dtype() == torch::kBFloat16 && vc.dtype() == torch::kBFloat16 &&
              kc.is_contiguous() && vc.is_contiguous() && bt.is_contiguous());
  TORCH_CHECK(out.dtype() == torch::kBFloat16 && out.size(0) == B && out.stride(1) == 1 &&
              dv <= DV && col + Hq * dv <= out.size(1));
  for (auto* t : {&slopes, &rates, &sink})
    TORCH_CHECK(!*t || ((*t)->numel() == Hq && (*t)->dtype() == torch::kFloat32));
  const HeadTurn ht = head_turn(turn, gate, slopes || rates, q, Hq, dv);
  TORCH_CHECK(ctx.numel() == B && bt.size(0) == B && bt.dtype() == torch::kInt32 &&
              ctx.dtype() == torch::kInt32);
  if (B == 0) return;
  auto* o = (__hip_bfloat16*)out.data_ptr() + col;
  const float* rp = rates ? rates->data_ptr<float>() : nullptr;
  const float* sp = slopes ? slopes->data_ptr<float>() : nullptr;
  const float* snk = sink ? sink->data_ptr<float>() : nullptr;
#define RUN1(DD, DVV, BB)                                                        \
  decode_launch<DD, DVV, false, BB>(q, kc, vc, bt, ctx, o, out.stride(0),        \
                                    (int)dv, (float)scale, (float)oscale,        \
                                    sp, rp, (int)window, (int)chunk, snk, ht, marks)
#define RUN(DD, DVV)                         \
  if (!sp) RUN1(DD, DVV, FLAT_BIAS);         \
  else if (rp) RUN1(DD, DVV, LOG_BIAS);      \
  else RUN1(DD, DVV, LINEAR_BIAS)
  if (D == 64 && DV == 64) { RUN(64, 64); }
  else if (D == 64 && DV == 128) { RUN(64, 128); }
  else if (D == 128 && DV == 64) { RUN(128, 64); }
  else if (D == 128 && DV == 128) { RUN(128, 128); }
  else TORCH_CHECK(false, "unsupported cache head widths ", D, ", ", DV);
#undef RUN
#undef RUN1
}
