// Flash-style causal prefill attention over the paged KV cache (gfx950).
//
// A wave owns 32 query rows of one head and computes S^T = K Q^T and O^T = V^T P^T
// (v_mfma_f32_32x32x16_bf16), so a lane owns one query row: maxima, sums and the
// rescaling of O are its own numbers and nothing of the softmax goes through LDS.
//  * P needs no exchange either: an accumulator of S^T holds keys 4 half + {0..3, 8..11}
//    of every 16, and V^T is read with its keys in just that order, four rows at a
//    time, by the transposing ds_read_b64_tr_b16.
//  * K and V tiles of 64 keys lie in LDS as they do in the cache, filled by
//    direct-to-LDS loads (an 8-bit cache goes through registers) into a ring of three
//    tiles: one barrier a tile, and a tile has a whole tile's computation to arrive.
//    16-byte units are XOR-swizzled by row, K's so that 16 rows of a column and V's so
//    that 4 neighbouring rows of 32 columns spread over the banks.
//  * The scores of the next 32 keys are computed among the exponentials of the current
//    ones, so the matrix cores and the vector unit work side by side within a wave.
//  * Weights are taken against a reference that need not be the maximum: it moves, and
//    O is rescaled, only when a score exceeds it by PRE_SLACK powers of two.
//
// What bounds it: 4096 rows behind 22000, 32 heads of 128 on 8 cached ones, keep the matrix
// units busy 54% of the cycles and the vector unit 50%; the clock falls to 1.9 GHz under
// them. 4135 us before (values transposed by 2-byte stores, nothing in flight, O rescaled
// through LDS), now 1480 us = 1090 TF/s; 4 x 2048 fresh rows 712 and 157 us = 877 TF/s;
// 8 x 800 fresh 230 and 74 us; heads of 64, 4 x 2048, 372 and 98 us; 8-bit cache, 2 x 2048
// behind 4000, 1070 and 363 us. Tried and slower: the values of a step delayed into the next
// one's exponentials (registers spill: 887 TF/s), a raised wave priority for the values.
//
// Geometry: 8 waves, HG = min(G, 4) query heads of ONE kv head x (8/HG)*32 query rows,
// so a staged tile serves all of them. Workgroups run through the head groups first:
// neighbours lie on different XCDs, and the workgroups of one XCD read the same heads'
// keys.
// BIAS adds a per-head distance penalty, linear, logarithmic or none, and a sliding
// window or chunks of positions (tiles and MFMA steps wholly outside of what a wave
// sees are skipped), lets keys and values differ in width, and writes scaled columns
// of a wider output. A sink starts every row's softmax from a term without key or
// value. EXTRA: GATED takes a sink and multiplies the head by a sigmoid gate; TAILED
// takes a key's last dimensions from a row that all heads share; TURNED turns the
// result back and gates its channels, in fp32 (head_turn.h).
// Covers fresh prefill and append-prefill (chunked agent turns) since K/V
// are read from the paged cache with an absolute-position causal bound.
#include "flash_tiles.h"
#include "head_turn.h"
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

#define CUR_STREAM c10::hip::getCurrentHIPStream().stream()

#define PRE_KEYS 64     // keys per tile
#define PRE_STAGES 3    // tiles in LDS
#define PRE_SLACK 10.f  // weights stay below 2^PRE_SLACK
enum { NO_BIAS = 0, LINEAR_BIAS = 1, LOG_BIAS = 2, FLAT_BIAS = 3 };
enum { PLAIN = 0, GATED = 1, TAILED = 2, TURNED = 3 };

// shared last dimensions of the keys: key t's are row t, its own come first in kc
struct KeyTail {
  const __hip_bfloat16* rows;
  long stride;
  int width;  // columns there are; the rest of D is zeros
  int own;    // dimensions in kc, a multiple of 8
};

// Few rows behind long contexts have fewer blocks than there are CUs, and a workgroup takes 1.6 us
// a tile of keys whatever the others do. The tiles of a block, unless they are few, are then cut
// into up to ``most`` parts, by a workgroup each, whose results [rows, heads, most, DV] and
// references and sums [.., 2] another kernel merges. 32 heads of 128 over 8, us, whole and cut:
// 100 rows behind 1500 45.8 and 27.5, behind 8000 199 and 37; 500 behind 1500 57.0 and 40.2, behind
// 8000 211 and 85; 1000 behind 8000 224 and 157; 4 of 60 behind 4000 106 and 45.
struct KeyCut {
  int most;
  float *part, *refs;
};
#define CUT_LEAST 6  // tiles of a part
// tiles of a part of a block that has n
DEVINL int part_tiles(int n, int most) {
  return n < 2 * CUT_LEAST ? 2 * CUT_LEAST : max(CUT_LEAST, (n + most - 1) / most);
}
// tiles of keys that the rows qoff.. of a block see
DEVINL int block_tiles(int qlen, int ctx, int qoff, int rows) {
  const int kend = min(ctx, ctx - qlen + qoff + min(qlen - qoff, rows));
  return (kend + PRE_KEYS - 1) / PRE_KEYS;
}

// HG: query heads per workgroup; PAGED: pages are whole tiles
template <int D, int DV, int HG, bool FP8, int BIAS, int EXTRA, bool PAGED, bool CUT = false>
__global__ __launch_bounds__(512, 1) void prefill_kernel(
    const __hip_bfloat16* __restrict__ q,   // [T, qstride], heads D apart
    const void* __restrict__ kc,  // [NP, Hkv, P, D] bf16 | fp8 e4m3
    const void* __restrict__ vc,
    __hip_bfloat16* __restrict__ out,       // [T, ostride], heads dv apart
    const int* __restrict__ block_seq,      // [NB] seq index of this q-block, or null:
    const int* __restrict__ block_qoff,     // [NB] q-row offset within the seq
    const int* __restrict__ cu_q, int S,    // [S+1]
    const int* __restrict__ block_tables,   // [S, MP]
    const int* __restrict__ ctx_lens,       // [S]
    int Hq, int Hkv, int P, int MP, float scale,
    long qstride, long ostride, int dv, float oscale,
    const float* __restrict__ slopes, const float* __restrict__ rates, int window,
    int chunk, const float* __restrict__ sink,  // [Hq], or null unless GATED
    const __hip_bfloat16* __restrict__ gate, long gstride,  // [T, gstride]
    KeyTail tail, HeadTurn turn, KeyCut cut) {
  static_assert(!CUT || (!BIAS && EXTRA == PLAIN));
  constexpr int NC = D / 16;        // Q^T fragments (MFMA K-chunks of K Q^T)
  constexpr int NDT = DV / 32;      // 32-wide d-tiles of O^T
  constexpr int KU = D / 8, VU = DV / 8;         // 16-B units of a key's, a value's row
  constexpr int LK = PRE_KEYS * KU / 512, LV = PRE_KEYS * VU / 512;  // loads per thread
  constexpr int KBYTES = PRE_KEYS * D * 2, STAGE = PRE_KEYS * (D + DV) * 2;
  // units of K's row r are XORed with (r >> KSHIFT) & KMASK; a row of 192 is one and a
  // half times 256 bytes, so pairs of rows share a permutation
  constexpr int KMASK = D == 128 ? 15 : 7, KSHIFT = D == 192 ? 1 : 0;
  constexpr int QS = 8 / HG;          // 32-row q sub-blocks per WG
  const int groups = Hq / HG;
  // late rows see most keys: first
  const int apart = CUT ? cut.most : 1, part = CUT ? blockIdx.x / groups % apart : 0;
  const int nb = gridDim.x / groups / apart - 1 - blockIdx.x / groups / apart;
  const int lane = threadIdx.x % WAVE;
  int seq, qoff;
  if (block_seq) {
    seq = block_seq[nb];
    qoff = block_qoff[nb];
  } else if (!find_block(cu_q, S, QS * 32, nb, lane, seq, qoff)) {
    return;
  }
  const int q_start = cu_q[seq];
  const int qlen = cu_q[seq + 1] - q_start;
  const int ctx = ctx_lens[seq];
  const int* bt = block_tables + (long)seq * MP;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int col = lane & 31;   // q column owned by this lane (within wave's 32)
  const int half = lane >> 5;  // half-wave
  // wave -> (query head, q sub-block): heads vary fastest so the HG heads
  // of one sub-block sit on consecutive waves
  const int h0 = blockIdx.x % groups * HG;
  const int h = h0 + (wave % HG);
  const int kvh = h0 / (Hq / Hkv);
  const int qsub = wave / HG;

  extern __shared__ __attribute__((aligned(16))) char smem[];
  const unsigned smem_at = (unsigned)(size_t)(__attribute__((address_space(3))) char*)smem;

  // ---- Q fragments (B operand of K Q^T): held for the whole block. A scale that is
  // not positive goes into them: the reference below compares unscaled scores
  const int qrow = qoff + qsub * 32 + col;  // local q row in this seq
  const bool qvalid = qrow < qlen;
  const long qbase = (q_start + (qvalid ? qrow : 0)) * qstride + (long)h * D;
  const unsigned flip = scale < 0.f ? 0x80008000u : 0u;
  const float c2 = scale == 0.f ? 1.f : fabsf(scale) * LOG2E;  // scores in units of log 2
  frag_u qf[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    bool there = qvalid && scale != 0.f;
    if constexpr (EXTRA == TAILED) there = there && c * 16 + half * 8 < tail.own + tail.width;
    if (there) {
      qf[c].s = *reinterpret_cast<const shortx8*>(q + qbase + c * 16 + half * 8);
#pragma unroll
      for (int k = 0; k < 4; ++k) qf[c].u[k] ^= flip;
    } else {
      qf[c].u[0] = qf[c].u[1] = qf[c].u[2] = qf[c].u[3] = 0u;
    }
  }

  const int q_abs = ctx - qlen + qrow;  // absolute position of this lane's q
  const bool has_sink = EXTRA == GATED || (BIAS && sink);
  // reference and this lane's part of the sum (its half of the keys)
  float m = has_sink ? fmaxf(sink[h] * LOG2E, -1e30f) : -1e30f;
  float l = has_sink && half == 0 ? 1.f : 0.f;
  floatx16 o[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;

  // keys needed by this q block: up to the last row's absolute position
  const int blk_rows = min(qlen - qoff, QS * 32);
  const int kend = min(ctx, ctx - qlen + qoff + blk_rows);
  int ntiles = (kend + PRE_KEYS - 1) / PRE_KEYS;
  bool whole = true;  // this workgroup sees all of the block's keys
  int from = 0;       // and the first tile it sees
  if constexpr (CUT) {
    const int per = part_tiles(ntiles, cut.most);
    from = part * per;
    whole = ntiles <= per;
    if (part > 0 && from >= ntiles) return;
    ntiles = min(ntiles, from + per);
  }
  // absolute position of the wave's first (smallest) q row
  const int q_abs_min = ctx - qlen + qoff + qsub * 32;

  // this head's penalty per token of distance, or per doubling of 1 + rate * distance,
  // in units of log 2; first key any row here sees
  const float slope = BIAS == LINEAR_BIAS ? slopes[h] * LOG2E
                      : BIAS == LOG_BIAS  ? slopes[h] : 0.f;
  const float rate = BIAS == LOG_BIAS ? rates[h] : 0.f;
  const int win = BIAS && window > 0 ? window : 0x3fffffff;
  // first key a query at position x sees (negative: all)
  auto first_seen = [&](int x) {
    const int lo = x - win + 1;
    return BIAS && chunk > 0 ? max(lo, x - x % chunk) : lo;
  };
  const int tile0 = BIAS ? max(0, first_seen(ctx - qlen + qoff)) / PRE_KEYS : from;
  const int lo = BIAS ? first_seen(q_abs) : 0;
  const int lo_max = BIAS ? first_seen(q_abs_min + 31) : 0;
  // tiles that the wave's rows see; the first of its workgroup's where there are no rows
  const bool rows = qoff + qsub * 32 < qlen;
  const int first = rows && BIAS ? max(first_seen(q_abs_min), 0) / PRE_KEYS : tile0;
  int end = rows ? (min(kend, q_abs_min + 32) + PRE_KEYS - 1) / PRE_KEYS : tile0;
  if constexpr (CUT) end = max(tile0, min(end, ntiles));

  // ---- tiles. A thread's unit x of a tile is unit tid + 512 x in LDS and takes what the
  // swizzle puts there. Pages are looked up a tile before the loads that need them (by
  // vector loads: with a scalar one under way every wait for LDS is for all of it); nothing
  // is computed from them until then, so nothing waits for them.
  constexpr int NP = PAGED ? 1 : D == DV ? LK : LK + LV;
  constexpr int EB = FP8 ? 1 : 2;  // bytes of a cached number
  int page[NP];
  auto key_column = [&](int x) {
    const unsigned row = (tid + x * 512u) / KU, slot = (tid + x * 512u) % KU;
    return (slot ^ ((row >> KSHIFT) & KMASK)) * 8;
  };
  auto value_column = [&](int x) {
    const unsigned row = (tid + x * 512u) / VU, slot = (tid + x * 512u) % VU;
    return (slot ^ (DV == 64 ? (row & 2) << 1 : (row & 3) << 2)) * 8;
  };
  auto unit_row = [&](int x) -> int {  // of K's units, then V's
    return x < LK ? (tid + x * 512u) / KU : (tid + (x - LK) * 512u) / VU;
  };
  const unsigned per = 0xffffffffu / P;  // t / P without a division
  auto page_of = [&](int t, int& in) {
    int pg = __umulhi((unsigned)t, per);
    in = t - pg * P;
    if (in >= P) { in -= P; ++pg; }
    return pg;
  };
  auto lookup = [&](int tile) {
    if (tile >= ntiles) return;
    int in;
    if constexpr (PAGED) {
      int at = page_of(tile * PRE_KEYS, in);
      asm("" : "+v"(at));
      page[0] = bt[at];
    } else {
#pragma unroll
      for (int x = 0; x < NP; ++x)
        page[x] = bt[page_of(min(tile * PRE_KEYS + unit_row(x), ctx - 1), in)];
    }
  };
  // Where unit x comes from, handed to ``load``. Past the end the last key stands again.
  // PAGED: the tile's place is a scalar and a thread's own offset is the same in all tiles
  // but the last.
  unsigned offset[2];  // of a thread's first unit of K and V; the others' rows follow
  constexpr int KSTEP = 512 / KU, VSTEP = 512 / VU;
  offset[0] = (unit_row(0) * D + key_column(0)) * EB;
  offset[1] = (unit_row(LK) * DV + value_column(0)) * EB;
  auto units = [&](int tile, auto load) {
    if constexpr (PAGED) {
      static_assert(512 % KU == 0 && KSTEP % 16 == 0 && VSTEP % 16 == 0);
      int in;
      page_of(tile * PRE_KEYS, in);
      const unsigned row =
          ((unsigned)__builtin_amdgcn_readfirstlane(page[0]) * Hkv + kvh) * P + in;
      const char* kt = (const char*)kc + (u64b)row * (D * EB);
      const char* vt = (const char*)vc + (u64b)row * (DV * EB);
      if (tile * PRE_KEYS + PRE_KEYS <= ctx) {
#pragma unroll
        for (int x = 0; x < LK; ++x) load(x, kt + x * KSTEP * D * EB + offset[0]);
#pragma unroll
        for (int x = 0; x < LV; ++x) load(LK + x, vt + x * VSTEP * DV * EB + offset[1]);
      } else {
        const int last = ctx - 1 - tile * PRE_KEYS;
#pragma unroll
        for (int x = 0; x < LK; ++x)
          load(x, kt + (unsigned)(min(unit_row(x), last) * D + key_column(x)) * EB);
#pragma unroll
        for (int x = 0; x < LV; ++x)
          load(LK + x, vt + (unsigned)(min(unit_row(LK + x), last) * DV + value_column(x)) * EB);
      }
    } else {
      // a cache holds fewer than 2^32 rows: it fits the card
      unsigned rows[NP], token[NP];
#pragma unroll
      for (int x = 0; x < NP; ++x) {
        int in;
        page_of(min(tile * PRE_KEYS + unit_row(x), ctx - 1), in);
        rows[x] = ((unsigned)page[x] * Hkv + kvh) * P + in;
        token[x] = (unsigned)page[x] * P + in;  // in a cache of one head
      }
#pragma unroll
      for (int x = 0; x < LK; ++x) {
        const unsigned d0 = key_column(x);
        const char* src = (const char*)kc + ((u64b)rows[x] * D + d0) * EB;
        if constexpr (EXTRA == TAILED) {
          // columns past the tail's are not there: the queries hold zeros for them
          const int past = (int)d0 - tail.own;
          if (past < 0) src = (const char*)kc + ((u64b)rows[x] * tail.own + d0) * EB;
          else if (tail.width > 0)
            src = (const char*)(tail.rows + token[x] * tail.stride +
                                (past < tail.width ? past : 0));
          else src = (const char*)kc + (u64b)rows[x] * tail.own * EB;
        }
        load(x, src);
      }
#pragma unroll
      for (int x = 0; x < LV; ++x)
        load(LK + x, (const char*)vc + ((u64b)rows[NP - LV + x] * DV + value_column(x)) * EB);
    }
  };
  auto issue = [&](int tile) {  // bf16: straight to LDS
    char* st = smem + (tile % PRE_STAGES) * STAGE + wave * 64 * 16;
    units(tile, [&](int x, const char* src) {
      char* dst = st + (x < LK ? x * 512 * 16 : KBYTES + (x - LK) * 512 * 16);
      __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)dst, 16, 0, 0);
    });
  };
  u64b u8[LK + LV];
  auto fetch8 = [&](int tile) {  // fp8: to registers, then (store8) converted to LDS
    units(tile, [&](int x, const char* src) { u8[x] = *reinterpret_cast<const u64b*>(src); });
  };
  auto store8 = [&](int tile) {
    char* st = smem + (tile % PRE_STAGES) * STAGE + tid * 16;
#pragma unroll
    for (int x = 0; x < LK + LV; ++x)
      *reinterpret_cast<shortx8*>(st + (x < LK ? x * 512 * 16 : KBYTES + (x - LK) * 512 * 16)) =
          fp8x8_to_bf16x8(u8[x]);
  };

  // ---- one step: 32 keys
  // this lane's K row (A operand: row col, contraction 8 half + j) and V^T addresses:
  // lane i of 16 reads 8 bytes of row i / 4; dt's columns move by 64 bytes
  // addresses in the tile at hand, K's one tile ahead; a tile's second step is a constant
  // further
  unsigned kat[NC], vat[NDT];
  {
    const int i = lane & 15, r = i >> 2;
    const int swz = DV == 64 ? (r & 2) << 1 : r << 2;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
      const int unit = dt * 4 + ((lane >> 4) & 1) * 2 + ((i & 3) >> 1);
      vat[dt] = smem_at + KBYTES + (4 * half + r) * DV * 2 + (unit ^ swz) * 16 + (i & 1) * 8;
    }
#pragma unroll
    for (int c = 0; c < NC; ++c)
      kat[c] = smem_at + col * D * 2 + (((c * 2 + half) ^ ((col >> KSHIFT) & KMASK)) << 4);
  }
  auto load_keys = [&](frag_u (&kf)[NC], int second, int from, int to) {
#pragma unroll
    for (int c = from; c < to; ++c)
      kf[c].s = *(const __attribute__((address_space(3))) shortx8*)(kat[c] + second * 32 * D * 2);
  };
  // O^T += V^T P^T, product j of 2 NDT: 16 keys j / NDT, d-tile j % NDT; fragments in pairs
  auto product = [&](const frag_u (&w)[2], const shortx4 (&v)[NDT][4], int j) {
    frag_u vf;
    vf.h[0] = v[j / 2][j % 2 * 2];
    vf.h[1] = v[j / 2][j % 2 * 2 + 1];
    o[j % NDT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf.v, w[j / NDT].v, o[j % NDT], 0, 0, 0);
  };
  // pair I of the step AT bytes into its tile
  auto fetch_values = [&](shortx4 (&v)[NDT][4], auto AT, auto I) {
    constexpr int i = decltype(I)::value, ROW8 = 8 * DV * 2;
    constexpr int at = decltype(AT)::value + i / (NDT / 2) * 2 * ROW8, dt = i % (NDT / 2) * 2;
    read_values<at, ROW8>(v[i], vat[dt], vat[dt + 1]);
  };
  using ZERO = std::integral_constant<int, 0>;
  using ONE = std::integral_constant<int, 1>;
  // penalty and mask of a step's scores
  auto mask = [&](floatx16& st, int step) {
    const int ks = step * 32;
    if constexpr (BIAS == LINEAR_BIAS || BIAS == LOG_BIAS) {
      // distance of key row 4 * half, and the logarithm's argument there
      const float dist0 = (float)(q_abs - ks - 4 * half);
      const float arg0 = 1.f + rate * dist0;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float away = (float)((r & 3) + 8 * (r >> 2));
        st[r] = st[r] * c2 - slope * (BIAS == LOG_BIAS ? __builtin_amdgcn_logf(arg0 - rate * away)
                                                       : dist0 - away);
      }
    }
    // (a row that has seen only masked keys yet keeps its first reference)
    if ((ks + 31 > q_abs_min) || (ks + 31 >= ctx) || (BIAS && ks < lo_max)) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int k_abs = ks + (r & 3) + 8 * (r >> 2) + 4 * half;
        if (k_abs > q_abs || k_abs >= ctx || (BIAS && k_abs < lo)) st[r] = -INFINITY;
      }
    }
  };

  // Softmax and values of ``step``, whose scores S^T (rows keys, columns queries) are in
  // ``cur``, and the scores of the step after it. A row's last step computes scores of
  // whatever lies in LDS, which nobody uses.
  auto advance = [&](floatx16& cur, floatx16& next, int step, auto SECOND) {
    constexpr bool SCALED = BIAS == LINEAR_BIAS || BIAS == LOG_BIAS;
    constexpr int second = decltype(SECOND)::value;
    using AT = std::integral_constant<int, second * 32 * DV * 2>;
    mask(cur, step);
    frag_u kf[NC];
    shortx4 v[NDT][4];
    constexpr int EARLY = NC < 8 ? NC : 8;  // the others when registers are free again
    load_keys(kf, 1 - second, 0, EARLY);
    float mx = cur[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, cur[r]);
    if constexpr (!SCALED) mx *= c2;
    if (__any(mx > m + PRE_SLACK)) {
      mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
      const float mn = fmaxf(m, mx);
      const float alpha = __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 16; ++r) next[r] = 0.f;
    frag_u pf[2];
    float sum = 0.f;
    // an eighth of the scores and of the softmax at a time
    static_for<8>([&](auto E) {
      constexpr int e = decltype(E)::value;
#pragma unroll
      for (int c = NC * e / 8; c < NC * (e + 1) / 8; ++c)
        next = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[c].v, qf[c].v, next, 0, 0, 0);
      float p[2];
#pragma unroll
      for (int k = 0; k < 2; ++k)
        p[k] = __builtin_amdgcn_exp2f(SCALED ? cur[2 * e + k] - m
                                             : __builtin_fmaf(cur[2 * e + k], c2, -m));
      sum += p[0] + p[1];
      pf[e >> 2].u[e & 3] = cvt2_bf16(p[0], p[1]);
      if constexpr (EARLY < NC && e == 2) load_keys(kf, 1 - second, EARLY, NC);
      if constexpr (e == 6) fetch_values(v, AT{}, ZERO{});
      __builtin_amdgcn_sched_barrier(0);
    });
    l += sum;
    await_values(v[0]);
    static_for<NDT>([&](auto I) {  // O^T += V^T P^T
      constexpr int i = decltype(I)::value;
      if constexpr (i + 1 < NDT) fetch_values(v, AT{}, std::integral_constant<int, i + 1>{});
      product(pf, v, 2 * i);
      product(pf, v, 2 * i + 1);
      if constexpr (i + 1 < NDT) await_values(v[i + 1]);
    });
  };

  // before and after the computation of a tile: the next one is there for all, and nobody
  // reads the one before it any more
  auto begin = [&](int tile) {
    if constexpr (FP8) {
      if (tile + 1 < ntiles) fetch8(tile + 1);
      lookup(tile + 2);
    }
  };
  auto turn_over = [&](int tile) {
    if constexpr (FP8) {
      if (tile + 1 < ntiles) store8(tile + 1);
      __syncthreads();
    } else {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (tile + 2 < ntiles) issue(tile + 2);
      lookup(tile + 3);
    }
  };
  // (a context shorter than its rows can leave a block without a key)
  if (tile0 < ntiles) {
    lookup(tile0);
    if constexpr (FP8) {
      fetch8(tile0);
      store8(tile0);
      lookup(tile0 + 1);
      __syncthreads();
    } else {
      issue(tile0);
      lookup(tile0 + 1);
      if (tile0 + 1 < ntiles) {
        issue(tile0 + 1);
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LK + LV) : "memory");
      } else {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      }
      lookup(tile0 + 2);
    }
  }
  int tile = tile0;
  for (; tile < first; ++tile) {
    begin(tile);
    turn_over(tile);
  }
  floatx16 even, odd;
  unsigned stage = tile % PRE_STAGES * STAGE;
#pragma unroll
  for (int c = 0; c < NC; ++c) kat[c] += stage;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) vat[dt] += stage;
  {  // the first scores
    frag_u kf[NC];
    load_keys(kf, 0, 0, NC);
#pragma unroll
    for (int r = 0; r < 16; ++r) even[r] = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c)
      even = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[c].v, qf[c].v, even, 0, 0, 0);
  }
  for (; tile < end; ++tile) {
    begin(tile);
    advance(even, odd, tile * 2, ZERO{});
    turn_over(tile);
    const unsigned move = stage == (PRE_STAGES - 1) * STAGE ? -(PRE_STAGES - 1) * STAGE : STAGE;
    stage += move;
#pragma unroll
    for (int c = 0; c < NC; ++c) kat[c] += move;
    advance(odd, even, tile * 2 + 1, ONE{});
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) vat[dt] += move;
  }
  for (; tile < ntiles; ++tile) {  // other waves' rows see more
    begin(tile);
    turn_over(tile);
  }

  // ---- epilogue: a lane holds channels 4 half + {0..3} of every 8 of its row
  l += __shfl_xor(l, 32, WAVE);
  const long row = q_start + qrow;
  if constexpr (CUT) {
    if (!whole) {
      if (!qvalid) return;
      const long at = (row * Hq + h) * cut.most + part;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<floatx4*>(cut.part + at * DV + dt * 32 + 8 * g + 4 * half) =
              floatx4{o[dt][4 * g], o[dt][4 * g + 1], o[dt][4 * g + 2], o[dt][4 * g + 3]};
      if (half == 0) *reinterpret_cast<floatx2*>(cut.refs + at * 2) = floatx2{m, l};
      return;
    }
  }
  if constexpr (EXTRA == GATED) {  // divided by l, times the gate
    const long grow = (q_start + (qvalid ? qrow : 0)) * gstride + h;
    l *= 1.f + __expf(-bf16_to_f32(((const unsigned short*)gate)[grow]));
  }
  const float inv = oscale / l;
  bf16_t* orow = (bf16_t*)out + row * ostride + (long)h * dv;
  const float* cs = EXTRA == TURNED && turn.cs ? turn.cs + (long)q_abs * dv : nullptr;
  const bf16_t* gp = EXTRA == TURNED && turn.gate
                         ? (const bf16_t*)turn.gate + row * turn.gstride + h * dv : nullptr;
  const bool vec = !BIAS || ((dv | ostride | ((long)out >> 1) |
                              (EXTRA == TURNED ? turn.gstride | ((long)turn.gate >> 1) : 0)) &
                             7) == 0;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) {
#pragma unroll
    for (int g = 0; g < 4; g += 2) {
      unsigned int y[2][2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int d = dt * 32 + 8 * (g + k) + 4 * half;
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = o[dt][4 * (g + k) + j] * inv;
        if constexpr (EXTRA == TURNED) {
          if (qvalid && d < dv) {
#pragma unroll
            for (int j = 0; j < 4; j += 2)
              if (cs && d + j < dv)
                turn_pair(v[j], v[j + 1], cs[(d + j) / 2], -cs[(dv + d + j) / 2]);
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (gp && d + j < dv) v[j] *= sigmoid_f(ldf(gp + d + j));
          }
        }
        if (!vec && qvalid) {  // head width or column not a multiple of 8
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (d + j < dv) stf(orow + d + j, v[j]);
        }
        y[k][0] = cvt2_bf16(v[0], v[1]);
        y[k][1] = cvt2_bf16(v[2], v[3]);
      }
      if (!vec) continue;
      // halves trade: this lane's half of 16 channels in one piece
      frag_u w;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const auto r = __builtin_amdgcn_permlane32_swap(y[0][j], y[1][j], false, false);
        w.u[j] = r[0];
        w.u[2 + j] = r[1];
      }
      const int d = dt * 32 + 8 * (g + half);
      if (qvalid && (!BIAS || d < dv)) *reinterpret_cast<shortx8*>(orow + d) = w.s;
    }
  }
}

// A row of every block whose keys were cut: its parts' results put together, a wave per head.
template <int DV>
__global__ __launch_bounds__(256) void merge_parts_kernel(
    KeyCut cut, __hip_bfloat16* __restrict__ out, const int* __restrict__ cu_q, int S,
    const int* __restrict__ ctx_lens, int Hq, int rows) {
  constexpr int N = DV / WAVE;
  const int row = blockIdx.x, lane = threadIdx.x % WAVE;
  const int h = blockIdx.y * 4 + threadIdx.x / WAVE;
  if (h >= Hq) return;
  int seq = 0;  // sequences that end before the row
  for (int s0 = 0; s0 < S; s0 += WAVE)
    seq += __popcll(__ballot(s0 + lane < S && cu_q[min(s0 + lane, S - 1) + 1] <= row));
  seq = __builtin_amdgcn_readfirstlane(seq);
  if (seq >= S) return;
  const int qlen = cu_q[seq + 1] - cu_q[seq], qoff = (row - cu_q[seq]) / rows * rows;
  const int n = block_tiles(qlen, ctx_lens[seq], qoff, rows), per = part_tiles(n, cut.most);
  if (n <= per) return;
  const int parts = (n + per - 1) / per;
  const long at = ((long)row * Hq + h) * cut.most;
  constexpr int AT_ONCE = 8;
  float o[AT_ONCE][N], y[N] = {};
  auto read = [&](int p0) {
#pragma unroll
    for (int k = 0; k < AT_ONCE; ++k)
#pragma unroll
      for (int j = 0; j < N; ++j)
        o[k][j] = cut.part[(at + min(p0 + k, parts - 1)) * DV + lane * N + j];
  };
  const floatx2 mine =
      *reinterpret_cast<const floatx2*>(cut.refs + (at + min(lane, parts - 1)) * 2);
  read(0);
  const float m = lane < parts ? mine[0] : -1e30f, M = wave_max(m);
  const float f = lane < parts ? __builtin_amdgcn_exp2f(m - M) : 0.f;
  const float inv = 1.f / wave_sum(f * mine[1]);
  for (int p0 = 0; p0 < parts; p0 += AT_ONCE) {
    if (p0 > 0) read(p0);
#pragma unroll
    for (int k = 0; k < AT_ONCE; ++k) {
      const float fp = __shfl(f, p0 + k, WAVE);
#pragma unroll
      for (int j = 0; j < N; ++j)
        if (p0 + k < parts) y[j] += fp * o[k][j];
    }
  }
  auto* dst = (unsigned short*)out + ((long)row * Hq + h) * DV + lane * N;
  if constexpr (N == 2) *reinterpret_cast<unsigned*>(dst) = cvt2_bf16(y[0] * inv, y[1] * inv);
  else dst[0] = f32_to_bf16(y[0] * inv);
}

// query heads per workgroup: the GQA group shares each staged K/V tile
static int heads_per_block(int G) { return G % 4 == 0 ? 4 : G % 2 == 0 ? 2 : 1; }

// A cache as loads straight to LDS can read it: 16-byte units at 16-byte addresses
static torch::Tensor unit_aligned(const torch::Tensor& cache) {
  const bool ok = (reinterpret_cast<uintptr_t>(cache.data_ptr()) & 15) == 0;
  return ok ? cache : cache.clone();
}

template <int D, int DV, int HG, bool FP8, int BIAS, int EXTRA, bool PAGED, bool CUT = false,
          typename... Args>
static void prefill_launch(const KeyCut& cut, int blocks, int Hq, Args... args) {
  constexpr int lds = PRE_STAGES * PRE_KEYS * (D + DV) * 2;
  const auto kern = prefill_kernel<D, DV, HG, FP8, BIAS, EXTRA, PAGED, CUT>;
  if (lds > 64 * 1024) {
    static const hipError_t once = hipFuncSetAttribute(
        (const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    TORCH_CHECK(once == hipSuccess, "attention prefill: LDS");
  }
  hipLaunchKernelGGL(kern, dim3(blocks * (CUT ? cut.most : 1) * (Hq / HG)), dim3(512), lds,
                     CUR_STREAM, args..., cut);
}

torch::Tensor attention_prefill_paged(torch::Tensor q, torch::Tensor kc,
                                      torch::Tensor vc, torch::Tensor bt,
                                      torch::Tensor cu_q, torch::Tensor ctx,
                                      double scale, c10::optional<torch::Tensor> into) {
  TORCH_CHECK(q.is_cuda() && q.dtype() == torch::kBFloat16, "bf16 GPU only");
  const int T = q.size(0), Hq = q.size(1), D = q.size(2);
  const int Hkv = kc.size(1), P = kc.size(2), MP = bt.size(1);
  TORCH_CHECK(D == 128 || D == 64, "head_dim must be 64 or 128, got ", D);
  auto out = result_like(q, into);
  if (T == 0) return out;
  kc = unit_aligned(kc);
  vc = unit_aligned(vc);
  TORCH_CHECK(Hq % Hkv == 0, "GQA requires Hq % Hkv == 0");
  const int HG = heads_per_block(Hq / Hkv);
  const int QROWS = 32 * (8 / HG);  // q rows covered per workgroup
  // as many blocks as there can be; each finds its rows, so that nothing is read back
  const int S = cu_q.numel() - 1, NB = T / QROWS + S;
  const bool fp8 = kc.dtype() == torch::kFloat8_e4m3fn;
  // A workgroup for every CU. The parts' way through memory and the merging take what is gained
  // of few tiles, the more the more blocks there are: 20 rows behind 700 (12 tiles, 8 blocks) 21.3
  // us whole and 18.1 cut, 300 behind 300 and 700 (10 and 16 tiles, 40 blocks) 23.7 and 29.1, 32.8
  // and 33.2, 500 behind 300 and 1000 (13 and 24, 64) 28.7 and 35.1, 45.9 and 38.0, 1000 behind 300,
  // 700 and 1500 (21, 27 and 40, 128) 40.8 and 47.6, 51.0 and 52.8, 70.5 and 63.8. (What the tables
  // have room for stands for the longest context; short ones of wide tables stay whole all the
  // same.) An 8-bit cache is not cut: the next layers' rows in it are made of these results, and
  // other sums let one in 20 to 50 of their bytes round the other way.
  const long blocks = (long)NB * (Hq / HG), least = 2 * CUT_LEAST + blocks / 8;
  KeyCut cut = {1, nullptr, nullptr};
  if (!fp8 && P % PRE_KEYS == 0 && (long)MP * P / PRE_KEYS >= least)
    cut.most = (int)std::max(1L, std::min(256 / blocks, 16L));
  torch::Tensor part, refs;
  if (cut.most > 1) {
    part = torch::empty({(long)T * Hq * cut.most * D}, q.options().dtype(torch::kFloat32));
    refs = torch::empty({(long)T * Hq * cut.most * 2}, q.options().dtype(torch::kFloat32));
    cut.part = part.data_ptr<float>(), cut.refs = refs.data_ptr<float>();
  }
#define PLAUNCH1(DD, HGV, F8, PG, CT)                                           \
  prefill_launch<DD, DD, HGV, F8, NO_BIAS, PLAIN, PG, CT>(cut, NB, Hq,             \
                     (const __hip_bfloat16*)q.data_ptr(),                     \
                     kc.data_ptr(), vc.data_ptr(),                            \
                     (__hip_bfloat16*)out.data_ptr(),                         \
                     nullptr, nullptr, cu_q.data_ptr<int>(), S, bt.data_ptr<int>(),                \
                     ctx.data_ptr<int>(), Hq, Hkv, P, MP, (float)scale,       \
                     (long)Hq * D, (long)Hq * D, D, 1.f, nullptr, nullptr, 0, \
                     0, nullptr, nullptr, 0, KeyTail{}, HeadTurn{})
#define PLAUNCH(DD, HGV)                                                      \
  if (cut.most > 1) {                                                         \
    PLAUNCH1(DD, HGV, false, true, true);                                     \
  } else if (P % PRE_KEYS == 0) {                                             \
    if (fp8) { PLAUNCH1(DD, HGV, true, true, false); }                        \
    else { PLAUNCH1(DD, HGV, false, true, false); }                           \
  } else if (fp8) { PLAUNCH1(DD, HGV, true, false, false); }                  \
  else { PLAUNCH1(DD, HGV, false, false, false); }
#define PLAUNCH_D(DD)                                                         \
  switch (HG) {                                                               \
    case 1: PLAUNCH(DD, 1); break;                                            \
    case 2: PLAUNCH(DD, 2); break;                                            \
    default: PLAUNCH(DD, 4); break;                                           \
  }
  if (D == 128) {
    PLAUNCH_D(128)
  } else {
    PLAUNCH_D(64)
  }
#undef PLAUNCH_D
#undef PLAUNCH
#undef PLAUNCH1
  HIP_CHECK_KERNEL();
  if (cut.most > 1) {
    const auto merge = D == 128 ? merge_parts_kernel<128> : merge_parts_kernel<64>;
    hipLaunchKernelGGL(merge, dim3(T, (Hq + 3) / 4), dim3(256), 0, CUR_STREAM, cut,
                       (__hip_bfloat16*)out.data_ptr(), cu_q.data_ptr<int>(), S,
                       ctx.data_ptr<int>(), Hq, QROWS);
    HIP_CHECK_KERNEL();
  }
  return out;
}

// query rows one workgroup of biased_attention_prefill covers
long biased_prefill_rows(long G) { return 32 * (8 / heads_per_block((int)G)); }

void biased_attention_prefill(torch::Tensor q, torch::Tensor kc, torch::Tensor vc,
                              torch::Tensor bt, torch::Tensor cu_q, torch::Tensor ctx,
                              torch::Tensor bseq, torch::Tensor boff, double scale,
                              long window, long chunk, c10::optional<torch::Tensor> slopes,
                              c10::optional<torch::Tensor> rates,
                              c10::optional<torch::Tensor> sink,
                              c10::optional<torch::Tensor> turn,
                              c10::optional<torch::Tensor> gate, torch::Tensor out,
                              long col, long dv, double oscale) {
  TORCH_CHECK(q.is_cuda() && q.dtype() == torch::kBFloat16 && q.is_contiguous());
  const int T = q.size(0), Hq = q.size(1), D = q.size(2);
  const int Hkv = kc.size(1), P = kc.size(2), MP = bt.size(1), DV = vc.size(3);
  TORCH_CHECK(Hq % Hkv == 0 && kc.size(3) == D && vc.size(1) == Hkv && vc.size(2) == P);
  TORCH_CHECK(kc.dtype() == torch::kBFloat16 && vc.dtype() == torch::kBFloat16 &&
              kc.is_contiguous() && vc.is_contiguous() && bt.is_contiguous());
  TORCH_CHECK(out.dtype() == torch::kBFloat16 && out.size(0) == T && out.stride(1) == 1 &&
              dv <= DV && col + Hq * dv <= out.size(1));
  for (auto* t : {&slopes, &rates, &sink})
    TORCH_CHECK(!*t || ((*t)->numel() == Hq && (*t)->dtype() == torch::kFloat32));
  const HeadTurn ht = head_turn(turn, gate, slopes || rates, q, Hq, dv);
  TORCH_CHECK(bseq.dtype() == torch::kInt32 && boff.dtype() == torch::kInt32 &&
              bseq.numel() == boff.numel() && cu_q.dtype() == torch::kInt32 &&
              cu_q.numel() == ctx.numel() + 1 && bt.size(0) == ctx.numel());
  const int NB = bseq.numel();
  if (T == 0 || NB == 0) return;
  kc = unit_aligned(kc);
  vc = unit_aligned(vc);
  const int HG = heads_per_block(Hq / Hkv);
  const float* rp = rates ? rates->data_ptr<float>() : nullptr;
  const float* sp = slopes ? slopes->data_ptr<float>() : nullptr;
  const float* snk = sink ? sink->data_ptr<float>() : nullptr;
#define BLAUNCH2(DD, DVV, HGV, BB, XX, PG)                                      \
  prefill_launch<DD, DVV, HGV, false, BB, XX, PG>(KeyCut{}, NB, Hq,                \
                     (const __hip_bfloat16*)q.data_ptr(), kc.data_ptr(),        \
                     vc.data_ptr(), (__hip_bfloat16*)out.data_ptr() + col,      \
                     bseq.data_ptr<int>(), boff.data_ptr<int>(),                \
                     cu_q.data_ptr<int>(), (int)ctx.numel(), bt.data_ptr<int>(), \
                     ctx.data_ptr<int>(), Hq, Hkv, P, MP, (float)scale,         \
                     (long)Hq * D, out.stride(0), (int)dv, (float)oscale,       \
                     sp, rp, (int)window, (int)chunk, snk, nullptr, 0, KeyTail{}, ht)
#define BLAUNCH1(DD, DVV, HGV, BB, XX)                                          \
  if (P % PRE_KEYS == 0) { BLAUNCH2(DD, DVV, HGV, BB, XX, true); }              \
  else { BLAUNCH2(DD, DVV, HGV, BB, XX, false); }
#define BLAUNCH(DD, DVV, HGV)                                                   \
  if (!sp) { BLAUNCH1(DD, DVV, HGV, FLAT_BIAS, TURNED); }           \
  else if (rp) { BLAUNCH1(DD, DVV, HGV, LOG_BIAS, PLAIN); }        \
  else { BLAUNCH1(DD, DVV, HGV, LINEAR_BIAS, PLAIN); }
#define BLAUNCH_HG(DD, DVV)                    \
  switch (HG) {                                \
    case 1: BLAUNCH(DD, DVV, 1); break;        \
    case 2: BLAUNCH(DD, DVV, 2); break;        \
    default: BLAUNCH(DD, DVV, 4); break;       \
  }
  if (D == 64 && DV == 64) { BLAUNCH_HG(64, 64) }
  else if (D == 64 && DV == 128) { BLAUNCH_HG(64, 128) }
  else if (D == 128 && DV == 64) { BLAUNCH_HG(128, 64) }
  else if (D == 128 && DV == 128) { BLAUNCH_HG(128, 128) }
  else TORCH_CHECK(false, "unsupported cache head widths ", D, ", ", DV);
#undef BLAUNCH_HG
#undef BLAUNCH
#undef BLAUNCH1
#undef BLAUNCH2
  HIP_CHECK_KERNEL();
}

// q [T, H, D] (rows may be strided), kc [NP, H, P, D], vc [NP, H, P, DV], gate
// [T, H] pre-activations (rows may be strided) -> out [T, H * DV]
void sink_attention_prefill(torch::Tensor q, torch::Tensor kc, torch::Tensor vc,
                            torch::Tensor bt, torch::Tensor cu_q, torch::Tensor ctx,
                            torch::Tensor bseq, torch::Tensor boff, double scale,
                            torch::Tensor sink, torch::Tensor gate, torch::Tensor out) {
  const int T = q.size(0), H = q.size(1), D = q.size(2);
  const int P = kc.size(2), MP = bt.size(1), DV = vc.size(3);
  TORCH_CHECK(q.is_cuda() && q.dtype() == torch::kBFloat16 && q.stride(2) == 1 &&
              q.stride(1) == D && q.stride(0) % 8 == 0 &&
              (reinterpret_cast<uintptr_t>(q.data_ptr()) & 15) == 0, "queries");
  TORCH_CHECK(kc.dtype() == torch::kBFloat16 && vc.dtype() == torch::kBFloat16 &&
              kc.is_contiguous() && vc.is_contiguous() && bt.is_contiguous() &&
              kc.size(1) == H && vc.size(1) == H && kc.size(3) == D && vc.size(2) == P &&
              vc.size(0) == kc.size(0), "keys and values");
  TORCH_CHECK(out.dtype() == torch::kBFloat16 && out.is_contiguous() && out.size(0) == T &&
              out.size(1) == (long)H * DV);
  TORCH_CHECK(gate.dtype() == torch::kBFloat16 && gate.size(0) == T && gate.size(1) == H &&
              gate.stride(1) == 1 && sink.numel() == H && sink.dtype() == torch::kFloat32);
  TORCH_CHECK(bseq.dtype() == torch::kInt32 && boff.dtype() == torch::kInt32 &&
              bseq.numel() == boff.numel() && cu_q.dtype() == torch::kInt32 &&
              bt.dtype() == torch::kInt32 && ctx.dtype() == torch::kInt32 &&
              cu_q.numel() == ctx.numel() + 1 && bt.size(0) == ctx.numel());
  const int NB = bseq.numel();
  if (T == 0 || NB == 0) return;
  kc = unit_aligned(kc);
  vc = unit_aligned(vc);
#define SLAUNCH(DD, DVV)                                                        \
  prefill_launch<DD, DVV, 1, false, NO_BIAS, GATED, false>(KeyCut{}, NB, H,         \
                     (const __hip_bfloat16*)q.data_ptr(), kc.data_ptr(),        \
                     vc.data_ptr(), (__hip_bfloat16*)out.data_ptr(),            \
                     bseq.data_ptr<int>(), boff.data_ptr<int>(),                \
                     cu_q.data_ptr<int>(), (int)ctx.numel(), bt.data_ptr<int>(), \
                     ctx.data_ptr<int>(), H, H, P, MP, (float)scale,            \
                     q.stride(0), out.stride(0), DV, 1.f, nullptr, nullptr, 0,  \
                     0, sink.data_ptr<float>(),                                 \
                     (const __hip_bfloat16*)gate.data_ptr(), gate.stride(0),    \
                     KeyTail{}, HeadTurn{})
  if (D == 64 && DV == 64) { SLAUNCH(64, 64); }
  else if (D == 64 && DV == 128) { SLAUNCH(64, 128); }
  else if (D == 128 && DV == 64) { SLAUNCH(128, 64); }
  else if (D == 128 && DV == 128) { SLAUNCH(128, 128); }
  else TORCH_CHECK(false, "unsupported head widths ", D, ", ", DV);
#undef SLAUNCH
  HIP_CHECK_KERNEL();
}

// q [T, H, D] (rows may be strided) against keys of which every head has ``own`` first
// dimensions in kc [NP, H, 1, own] and all heads share the others, tail [NP, n] (rows
// may be strided; zeros follow up to D); vc [NP, H, 1, DV] -> out [T, H * DV]
void tailed_attention_prefill(torch::Tensor q, torch::Tensor kc, torch::Tensor vc,
                              torch::Tensor tail, torch::Tensor bt, torch::Tensor cu_q,
                              torch::Tensor ctx, torch::Tensor bseq, torch::Tensor boff,
                              double scale, long window, torch::Tensor out) {
  const int T = q.size(0), H = q.size(1), D = q.size(2);
  const int MP = bt.size(1), DV = vc.size(3), own = kc.size(3);
  TORCH_CHECK(q.is_cuda() && q.dtype() == torch::kBFloat16 && q.stride(2) == 1 &&
              q.stride(1) == D && q.stride(0) % 8 == 0 &&
              (reinterpret_cast<uintptr_t>(q.data_ptr()) & 15) == 0, "queries");
  TORCH_CHECK(kc.dtype() == torch::kBFloat16 && vc.dtype() == torch::kBFloat16 &&
              kc.is_contiguous() && vc.is_contiguous() && bt.is_contiguous() &&
              kc.size(1) == H && vc.size(1) == H && kc.size(2) == 1 && vc.size(2) == 1 &&
              own < D && own % 8 == 0 && vc.size(0) == kc.size(0), "keys and values");
  TORCH_CHECK(tail.dtype() == torch::kBFloat16 && tail.dim() == 2 && tail.stride(1) == 1 &&
              tail.size(0) == kc.size(0) && tail.size(1) % 8 == 0 &&
              tail.stride(0) % 8 == 0 &&
              (reinterpret_cast<uintptr_t>(tail.data_ptr()) & 15) == 0, "shared key part");
  TORCH_CHECK(out.dtype() == torch::kBFloat16 && out.is_contiguous() && out.size(0) == T &&
              out.size(1) == (long)H * DV);
  TORCH_CHECK(bseq.dtype() == torch::kInt32 && boff.dtype() == torch::kInt32 &&
              bseq.numel() == boff.numel() && cu_q.dtype() == torch::kInt32 &&
              bt.dtype() == torch::kInt32 && ctx.dtype() == torch::kInt32 &&
              cu_q.numel() == ctx.numel() + 1 && bt.size(0) == ctx.numel());
  const int NB = bseq.numel();
  if (T == 0 || NB == 0) return;
  kc = unit_aligned(kc);
  vc = unit_aligned(vc);
  const KeyTail kt = {(const __hip_bfloat16*)tail.data_ptr(), tail.stride(0),
                      (int)tail.size(1), own};
#define TLAUNCH(DD, DVV)                                                        \
  prefill_launch<DD, DVV, 1, false, FLAT_BIAS, TAILED, false>(KeyCut{}, NB, H,       \
                     (const __hip_bfloat16*)q.data_ptr(), kc.data_ptr(),        \
                     vc.data_ptr(), (__hip_bfloat16*)out.data_ptr(),            \
                     bseq.data_ptr<int>(), boff.data_ptr<int>(),                \
                     cu_q.data_ptr<int>(), (int)ctx.numel(), bt.data_ptr<int>(), \
                     ctx.data_ptr<int>(), H, H, 1, MP, (float)scale,            \
                     q.stride(0), out.stride(0), DV, 1.f, nullptr, nullptr,     \
                     (int)window, 0, nullptr, nullptr, 0, kt, HeadTurn{})
#define TLAUNCH_D(DD)                       \
  if (D == DD && DV == 64) { TLAUNCH(DD, 64); } \
  else if (D == DD && DV == 128) { TLAUNCH(DD, 128); } else
  TLAUNCH_D(64) TLAUNCH_D(128) TLAUNCH_D(192)
  TORCH_CHECK(false, "unsupported head widths ", D, ", ", DV);
#undef TLAUNCH_D
#undef TLAUNCH
  HIP_CHECK_KERNEL();
}
