// Which products the own kernels take: the one place where a call of x @ w^T is decided, in
// native code because a layer makes four such calls and an eager step has some 5 us for each
// (the same rules in Python, asked again by each form, took 4 to 8 us a product, this 1).
#include "plain.h"
#include <c10/core/DeviceGuard.h>
#include <cstdlib>
#include <cstring>

// defined in few_rows.hip, moe.hip, skinny_gemm.hip
torch::Tensor linear_few_rows(torch::Tensor x, torch::Tensor w, bool raw, bool steady);
torch::Tensor silu_few_rows(torch::Tensor x, torch::Tensor w);
torch::Tensor block_rows(torch::Tensor x, torch::Tensor w, bool raw);
int block_form(long M, long N, long K, bool raw);
bool one_row_fits(long S, long K);
bool float_few_rows_fits(long N, long K);
torch::Tensor float_few_rows(torch::Tensor x, torch::Tensor w);
torch::Tensor many_rows(torch::Tensor x, torch::Tensor w, bool silu);
bool large_takes(long N, long K);
torch::Tensor skinny_gemm3_ex(torch::Tensor x, torch::Tensor w, long s_target);

// STEADY beside a form: what the rows of prompts go through on their way into an 8-bit cache. They
// are most of its bytes, and sums in another order let one in 20 to 50 of those round the other
// way, so such products stay where, and in the parts of K in which, they were first made.
enum { WHOLE = 0, PARTS = 1, SILU = 2, FLOAT = 3, STEADY = 4 };

static long megabytes(long N, long K) { return (N * K * 2) >> 20; }

// Weights up to here are read in one go by the kernel of few rows, whatever their shape.
static long small_megabytes() {
  const char* mb = std::getenv("AURORA_SKINNY_MAX_MB");
  return mb ? std::atol(mb) : 128;
}

// Up to 128 rows: where the kernel beats the library's. us with cold weights, ours and the
// library's. Small weights up to 64 rows (4096 x 14336, 23 rows 24 and 33). Larger ones up to
// 32 rows while K is short, up to 512 MB of them to 4096 (1 and 32 rows: 152064 x 3584 195
// and 233, 208 and 264; 32000 x 4096 54 and 60, 56 and 66; but 128256 x 4096 204 and 187, 207
// and 201; 57344 x 8192 213 and 181; 16384 x 8192 66 and 62, 65 and 54; the other way, given
// up, 28672 x 8192 105 and 131). Few outputs of long K, which is cut, whatever their size (1, 32
// and 64 rows with the norm that reads them: 3584 x 18944 30 and 52, 32 and 113, 33 and 94; 5120 x
// 27648 56 and 141, 56 and 153, 60 and 163; 7168 x 18432 59 and 57, 54 and 61, 58 and 130; 8192 x
// 28672 96 and 94, 87 and 100, 93 and 142; 10240 x 8192 44 and 42, 41 and 45, 42 and 49; without
// it 7168 x 18432, 16 and 64 rows, 53 and 110, 56 and 124). Above 64 rows up to 12288 outputs with
// parts that their reader adds up (3072 x 2048, 96 rows, 8 and 13; with a norm 9216 x 4096 27 and
// 35, 10240 x 8192 44 and 58, 12288 x 4096 32 and 38; but 16384 x 4096 44 and 44), or up to 8192
// with K long enough to pay for adding them, few outputs with longer ones (96 rows: 4608 x 4096 16
// and 22, 2048 x 4096 13.3 and 12.8, 2048 x 8192 15 and 21, 1024 x 8192 15.2 and 15.0, 1024 x 14336
// 17 and 25, 8192 x 28672 123 and 124; but 4608 x 2048 13.1 and 13.5, 128 rows 15.9 and 15.0; 10240
// x 8192 57 and 55).
static bool few_rows_win(long M, long N, long K, bool parts, bool steady) {
  if (M > 64)
    return N <= (parts && !steady ? 12288 : 8192) &&
           (parts || K >= 14336 || (K >= 3072 && N >= (K < 8192 ? 3072 : 2048)));
  const long size = megabytes(N, K);
  const long most = M == 1 ? 6144 : !parts ? 7168 : M <= 32 ? 8192 : 10240;
  return size <= small_megabytes() || (K > 4096 && N <= most && !steady) ||
         (M <= 32 && (K < 4096 || (K == 4096 && size <= 512)));
}

// The same with silu, N outputs of 2 N rows of weights, against a library product and an
// activation: K is not cut here, so a tile of 32 outputs takes its K's time and long K wants
// tiles for all CUs, above 32 rows as many for each (``even``). Library's time over ours at
// 1, 23, 64, 96 and 128 rows:
//   K     tiles 16                  56                       112
//   2048  1.25 1.26 0.93 0.75 0.60  1.23 1.24 1.01 1.02 0.90  1.20 1.20 1.01 1.05 0.92
//   3072  1.18 1.11 0.79 0.58 0.47  1.17 0.99 0.80 0.73 0.65  1.05 0.96 1.00 0.91 0.84
//   4096  0.80 0.82 0.70 0.54 0.43  0.84 0.83 0.66 0.60 0.54  1.02 0.94 0.87 0.89 0.76
//   8192  0.51 0.51 0.42 0.36 0.28  0.66 0.68 0.54 0.47 0.43  0.83 0.79 0.78 0.78 0.67
//         tiles 160                 224                      296
//   2048  1.17 1.16 1.16 1.08 1.01  1.11 1.15 1.13 1.15 0.97  1.09 1.11 1.03 1.07 0.96
//   3072  1.13 1.10 1.09 1.10 0.97  1.08 1.12 1.05 1.08 1.03  1.08 1.02 0.98 0.87 0.79
//   4096  1.04 1.06 1.08 1.09 0.95  1.02 1.05 0.98 1.07 0.97  1.02 0.99 0.93 0.86 0.79
//   8192  0.93 0.98 0.90 0.99 0.89  0.91 0.94 0.90 1.01 0.91  0.86 1.01 0.87 0.83 0.75
// K 1024 1.05 to 1.55, but 0.95 at 16 tiles and 128 rows; 4096 with 448 tiles 1.40 1.21 1.07
// 1.02 1.01, with 384 1.05 1.07 0.96 1.01 0.97; 3584 with 592 1.03 1.04 1.00 0.89 0.84; 8192
// with 896 0.96 0.92 0.94 1.00 0.98.
static bool silu_few_rows_win(long M, long N, long K) {
  const long tiles = (N + 31) / 32;
  const bool even = tiles <= 256 || (tiles >= 410 && tiles <= 512);
  if (K <= 1024) return true;
  if (M <= 32)
    return K <= 3072 || (K <= 4096 && tiles >= 88) || (K <= 5120 && tiles >= 160);
  if (M <= 64)
    return K <= 3072 ? tiles >= (K <= 2048 ? 32 : 88) : K <= 4096 && tiles >= 160 && even;
  if (M <= 96) return K <= 2048 ? tiles >= 56 : K <= 4096 && tiles >= 160 && even;
  return K <= 2048 && tiles >= 160;
}

// More than 128 rows: where the kernel of 256-row tiles beats the library's product (with
// silu, product and activation). A CU has one tile at a time and K is not cut, so what counts
// is for how many of the 256 CUs there is work, in tiles of 128 rows x 256 rows of w. Library's
// time over ours by them, cold weights, means of sizes from 129 to 8192 rows and 16 to 57344
// rows of w (least from 256 tiles on). With silu:
//   K to   8     16    24    40    56    72    96    120   144   176   208   256
//   512    1.09  1.22  1.29  1.42  1.53  1.75  1.70  1.82  1.86  1.89  2.07  2.18 (1.61)
//   1024   0.94  1.00  1.03  1.13  1.21  1.29  1.34  1.39  1.44  1.42  1.39  1.43 (1.05)
//   2048   0.66  0.72  0.79  0.91  0.96  1.08  1.08  1.12  1.18  1.17  1.17  1.20 (0.87)
//   4096   0.49  0.57  0.62  0.71  0.77  0.87  0.88  0.98  1.07  1.04  1.07  1.13 (0.81)
//   8192   0.36  0.42  0.51  0.62  0.71  0.84  0.78  0.91  1.01  0.95  1.02  1.06 (0.75)
// What falls behind beyond the lines are 192 and 256 rows (not 208, 224 or 240) of 33000 to
// 43500 rows of w, K above 1024 (0.75 to 1.04); 44000 to 49000 of them, 264 to 512 rows, K from
// 3072 on are even (0.90 to 1.15). Without silu:
//   K to   16    24    40    72    96    120   144   176   200   224   256
//   512    0.88  0.97  1.08  1.20  1.18  1.21  1.33  1.30  1.67  1.32  1.46 (1.00)
//   1024   0.78  0.83  0.90  0.97  0.98  1.01  1.09  1.11  1.16  1.11  1.18 (0.95)
//   2048   0.57  0.66  0.81  0.90  0.94  0.97  1.04  1.04  1.13  1.10  1.12 (0.90)
//   4096   0.50  0.57  0.70  0.76  0.81  0.89  0.97  0.97  1.06  1.05  1.09 (0.92)
//   8192   0.38  0.47  0.63  0.69  0.74  0.82  0.89  0.93  1.00  1.02  1.05 (0.90)
//   28672  0.42  0.53  0.71  0.72  0.77  0.84  0.94  0.93  1.52  1.04  1.16 (0.93)
// (K up to 256 0.90 from 24, 0.96 from 32), but whole rounds of the library's own tiles of 256 x
// 256 are its (K above 1024 0.90 to 1.02), and long K wants tiles well filled (129 rows of 28672 x
// 4096 0.85, with silu 0.90, 160 rows 0.93, 192 rows 0.97). In either form the library
// falls behind at up to 256 rows of x and of w while K is short (K to 832 0.97 to 3.6), and keeps
// long K where no round counts any more (140000 rows, 8192 x 8192 with silu 0.96, 4096 x 8192
// without 0.95; but 300000, 4096 x 4096 1.06, 2048 x 4096 1.02; 600000, 2048 x 2048 1.22).
static bool many_rows_win(long M, long N, long K, bool silu) {
  const long tiles = (M + 127) / 128 * N / 256, cols = (N + 255) / 256;
  if (M <= 256 && N <= 256 && K <= 832) return true;
  if (K > 4096 && tiles >= 16384) return false;
  if (silu) {
    if (K > 1024 && M <= 256 && M % 64 == 0 && cols > 128 && cols <= 170) return false;
    if (K > 2048 && M <= 256 && M * N < 160 * 128 * 256) return false;
    return K <= 512 || tiles >= (K <= 1024 ? 24 : K <= 2048 ? 72 : K <= 4096 ? 144 : 208);
  }
  if (K > 1024 && M % 256 == 0 && N % 256 == 0 && M / 256 * cols % 256 == 0) return false;
  if (K > 2048) return tiles >= 200 && M * N >= 176 * 128 * 256;
  return tiles >= (K <= 256 ? 40 : K <= 512 ? 24 : K <= 1024 ? 120 : 144);
}

// AURORA_SKINNY3=0 leaves 192 to 256 rows to the library.
static bool left_to_library(long M) {
  if (M < 192 || M > 256) return false;
  const char* off = std::getenv("AURORA_SKINNY3");
  return off && !std::strcmp(off, "0");
}

// 65 to 1000 rows: where the kernel of few rows, in blocks of rows, beats the library's product.
// us with cold weights, the library's and ours, whole and in parts with the norm that reads them:
//   N x K         rows: 140            256            300            512            1000
//   4096 x 4096     22 18, 26 19   23 23, 27 23   26 26, 30 27   30 30, 35 35   43 43, 50 50
//   6144 x 4096     39 25, 44 26   37 28, 41 32   29 30, 35 35   38 38, 45 44   54 54, 64 63
//   4096 x 14336    57 40, 60 40   62 48, 67 49   75 67, 80 67   93 82, 97 84   141 141, 150 148
//   2048 x 2048     12 11, 15 11   12 12, 15 13   13 12, 16 14   13 13, 17 16   17 16, 22 21
//   2048 x 8192     26 18, 30 20   27 22, 31 23   33 25, 37 26   35 32, 38 33   52 52, 57 51
//   768 x 768      6.8 5.7, 10 8  6.8 5.6, 10 8  6.8 5.7, 10 8  7.2 5.8, 11 9  7.5 5.9, 11 10
//   768 x 3072     9.5 9.6, 13 10  10 11, 14 11   10 12, 13 12   15 12, 19 13   17 17, 20 18
//   2304 x 768     9.5 6.2, 13 9  9.7 6.6, 13 10 9.8 6.6, 14 10  10 7.3, 15 12  13 13, 18 18
// and a call of the library's takes the host 11 to 15 us more, which small prompts and texts wait
// for (a text of 200 tokens 1197 us and 612). The line is work for a quarter of the chip, in tiles
// of 128 x 256: beyond it both come to the same by themselves (with the norm 520 rows of 4096 x
// 4096 39 and 36, of 4096 x 14336 111 and 111, 768 of 3584 x 14336 113 and 127) and four layers of
// 4096, 520 rows, took 1647 and 1746 us. In front of it, more than 256 rows of K 2560 to 8192 take
// as long as the library's where they come whole in one round of workgroups with a tile's blocks
// on one or two XCDs (0.86 to 1.09, mean of 348 sizes 1.00; 512 rows of 4096 x 4096 28.5 and 29.5
// us); on four XCDs 1.03 times as long, on eight 1.10, in more rounds 1.11 (512 rows of 2816 x 5632
// 37.5 and 33.6, 1000 of 1536 x 5632 37.7 and 32.4). Cut for a reader who does not add the parts
// up they take 1.00 to K 6144 and 0.96 beyond. Of 3084 sizes within the lines ours takes 0.83 of
// the library's time whole, 0.79 with the norm. What falls behind by more than 4% are whole
// products of 512 to 1536 outputs, K of 1400 to 3100 (10 us where the library takes 9, and the
// host 20: 512 x 1408 8.5 and 9.1, 1408 x 2816, 140 rows, 9.8 and 11.3, 768 x 3072, 300 rows, 10.0
// and 11.9).
// 65 to 128 rows, whole (few_rows_win has those in parts), 65, 96 and 128, the library's and ours:
//   K      1024 outputs                2304                        2560
//   768    9.1 6.1, 9.0 6.2, 8.9 6.5   9.0 6.1, 9.2 6.2, 10 6.5    9.1 6.2, 9.1 6.3, 10 6.7
//   1408   8.3 8.2, 8.7 8.8, 8.6 9.2   8.3 8.8, 8.9 8.9, 15 9.3    9.0 8.9, 9.1 9.0, 15 9.5
//   2048   11 8.6, 11 9.6, 11 9.5      11 9.7, 11 10, 14 11        11 9.9, 11 10, 14 11
//          2816                        4096                        8192
//   768    9.6 6.2, 9.9 6.3, 10 6.6    9.6 6.4, 10 6.4, 10 6.7     10 6.6, 10 6.8, 11 7.1
//   1408   9.7 8.9, 10 9.0, 15 9.3     9.6 9.1, 10 9.1, 15 9.6     11 9.7, 11 9.8, 16 10
//   2048   12 11, 13 11, 15 11         12 11, 13 12, 15 12         14 13, 14 13, 16 13
// where ours is ahead from 2816 outputs on at every K. (Fewer, down to 2304, are even at 1408 and
// ahead beside it; 1024 falls behind there.)
// K up to 512: 256 x 256 9.2 3.8, 8.4 3.5, 7.9 3.6, 4096 x 256 5.8 3.9, 6.1 4.2, 6.8 4.3, 1024 x
// 512 7.3 4.7, 6.5 4.5, 7.7 4.5 (65, 100 and 128 rows).
static bool block_rows_win(long M, long N, long K, bool parts) {
  if (left_to_library(M)) return false;
  if (M <= 128) return N <= 8192 && (K <= 512 ? N >= 64 : K <= 2048 && N >= 2816);
  const long work = (M + 127) / 128 * N / 256;  // (a little more, many_rows takes)
  if (K <= 512) return M <= 1000 && N >= 64 && work <= (K <= 256 ? 40 : 16);
  if (M > 1000 || N < 512 || (M + 127) / 128 * N > 64 * 256) return false;
  if (M <= 256 || K <= 2048 || work < 44) return true;
  const int form = block_form(M, N, K, parts);
  return form == 1 || (form == 2 && (parts || K > 8192));
}

// x @ w^T in ``form``, or nothing: the library's product serves better or is followed by
// autograd, a transform or a trace, or the kernels have no form for it.
c10::optional<torch::Tensor> own_product(const torch::Tensor& x, const torch::Tensor& w,
                                         long asked) {
  const long form = asked & ~STEADY;
  const bool steady = asked & STEADY;
  if (!plain(x) || !plain(w) || x.dim() != 2 || w.dim() != 2 || !x.is_cuda() ||
      x.device() != w.device() || x.dtype() != torch::kBFloat16 ||
      w.dtype() != torch::kBFloat16)
    return {};
  const long M = x.size(0), K = x.size(1), N = w.size(0);
  if (M == 0 || K == 0 || K % 64 || K != w.size(1) || !w.is_contiguous() ||
      (uintptr_t)w.data_ptr() % 16 || (x.is_contiguous() && (uintptr_t)x.data_ptr() % 16))
    return {};
  const c10::DeviceGuard on(x.device());
  if (form == SILU) {
    if (N % 16) return {};
    if (M <= 128) {
      if (!silu_few_rows_win(M, N / 2, K)) return {};
      return silu_few_rows(x, w);
    }
    if (large_takes(N, K) && many_rows_win(M, N, K, true))
      return many_rows(x, w, true);
    return {};
  }
  if (form == FLOAT) {
    // (of more than 64 rows none that few_rows_win names has its K whole)
    if (M > 64 || !few_rows_win(M, N, K, false, steady) || !float_few_rows_fits(N, K)) return {};
    return float_few_rows(x, w);
  }
  if (M <= 128) {
    if (form == PARTS && few_rows_win(M, N, K, true, steady))
      return linear_few_rows(x, w, true, steady);
    if (few_rows_win(M, N, K, false, steady)) return linear_few_rows(x, w, false, steady);
    if (!steady && M > 64 && block_rows_win(M, N, K, form == PARTS))
      return block_rows(x, w, form == PARTS);
  } else if (large_takes(N, K) && many_rows_win(M, N, K, false)) {
    return many_rows(x, w, false);
  } else if (steady) {
    if (M >= 192 && M <= 256 && N % 64 == 0 && N > 4096 && N <= 6144 && K > 2048 && K <= 4096 &&
        !left_to_library(M))
      return skinny_gemm3_ex(x.contiguous(), w, 384);
  } else if (block_rows_win(M, N, K, form == PARTS)) {
    return block_rows(x, w, form == PARTS);
  }
  return {};
}

// Whether the norm of x's parts + res by ``weight`` is done by the product with w that reads it,
// in parts or with ``silu``: one row, where the kernel of few rows would take the product.
bool norms_row(const torch::Tensor& x, const torch::Tensor& res, const torch::Tensor& weight,
               const torch::Tensor& w, bool silu, bool steady) {
  if (x.dim() != 3 || x.size(1) != 1 || x.dtype() != torch::kFloat32 || !x.is_cuda() ||
      !plain(x) || !x.is_contiguous() || (uintptr_t)x.data_ptr() % 16)
    return false;
  const long K = x.size(2);
  for (const auto* t : {&res, &weight, &w})
    if (!plain(*t) || t->device() != x.device() || t->dtype() != torch::kBFloat16 ||
        !t->is_contiguous() || (uintptr_t)t->data_ptr() % 16)
      return false;
  if (!one_row_fits(x.size(0), K) || res.dim() != 2 || res.size(0) != 1 || res.size(1) != K ||
      weight.numel() != K || w.dim() != 2 || w.size(1) != K || w.size(0) == 0 || w.size(0) % 16)
    return false;
  return silu ? silu_few_rows_win(1, w.size(0) / 2, K)
              : few_rows_win(1, w.size(0), K, true, steady);
}
