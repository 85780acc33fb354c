// Which products the own kernels take: the one place where a call of x @ w^T is decided, in
// native code because a layer makes four such calls and an eager step has some 5 us for each
// (the same rules in Python, asked again by each form, took 4 to 8 us a product, this 1).
#include "plain.h"
#include <c10/core/DeviceGuard.h>
#include <cstdlib>
#include <cstring>

// defined in few_rows.hip, moe.hip, skinny_gemm.hip
torch::Tensor linear_few_rows(torch::Tensor x, torch::Tensor w, bool raw);
torch::Tensor silu_few_rows(torch::Tensor x, torch::Tensor w);
torch::Tensor many_rows(torch::Tensor x, torch::Tensor w, bool silu);
torch::Tensor skinny_gemm3_ex(torch::Tensor x, torch::Tensor w, long s_target);

enum { WHOLE = 0, PARTS = 1, SILU = 2 };

// Up to 128 rows, where the kernel beats the library's (us, cold weights): up to 32 rows
// always (28672 x 4096, 23 rows 50 and 56, 128256 x 2048 101 and 120); up to 64 while the
// weights are at most 128 MB (16384 x 2048 18 and 19, but 37888 x 3584 66 and 62); above that
// up to 8192 outputs with parts that their reader adds up (3072 x 2048, 96 rows, 8 and 13),
// or with K long enough to pay for adding them (4096 x 4096 15 and 22, 6144 x 4096 22 and 23,
// but 2048 x 2048 11 and 9).
static bool few_rows_win(long M, long N, long K, bool parts) {
  if (M <= 32) return true;
  if (M <= 64) {
    const char* mb = std::getenv("AURORA_SKINNY_MAX_MB");
    return N * K * 2 <= (mb ? std::atol(mb) : 128) * 1024 * 1024;
  }
  return N <= 8192 && (parts || K >= 3072);
}

// More than 128 rows, where the kernel of 256-row tiles beats the library's product (with
// silu, product and activation), us. With silu: any number of tiles up to 1024 of K (6144 x
// 768, 300 rows 22 and 25, 27000 rows 250 and 349), else those that fill the chip's rounds
// (16384 x 2048, 600 rows 45 and 48, 6172 rows 330 and 411; 28672 x 4096, 2048 rows 371 and
// 376, 6172 rows 1132 and 1224; not full: 1600 rows 346 and 341, 12288 x 4096, 3000 rows 255
// and 248). Without: only where the tiles nearly fill the chip twice and K is long, where the
// library falls to 0.75 to 1.2 PFLOP/s (4096 x 14336, 6172 rows 594 and 807, 7000 rows 630 and
// 696; 3584 x 18944, 7500 rows 798 and 1184; outside: 6144 rows of 4096 x 14336 586 and 565,
// 8000 rows 677 and 629).
static bool many_rows_win(long M, long N, long K, bool silu) {
  const long tiles = (M + 255) / 256 * ((N + 255) / 256), rounds = (tiles + 255) / 256;
  if (!silu) return K >= 14336 && tiles > 384 && tiles < 512;
  if (K <= 1024) return M >= 256 && tiles >= 48;
  return tiles >= 192 && tiles >= (K <= 2048 ? 0.75 : 0.78) * 256 * rounds;
}

// x @ w^T in ``form``, or nothing: the library's product serves better or is followed by
// autograd, a transform or a trace, or the kernels have no form for it.
c10::optional<torch::Tensor> own_product(const torch::Tensor& x, const torch::Tensor& w,
                                         long form) {
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
    if (M <= 128) return silu_few_rows(x.contiguous(), w);
    if (many_rows_win(M, N, K, true)) return many_rows(x.contiguous(), w, true);
    return {};
  }
  if (M <= 128) {
    if (form == PARTS && few_rows_win(M, N, K, true))
      return linear_few_rows(x.contiguous(), w, true);
    if (few_rows_win(M, N, K, false)) return linear_few_rows(x.contiguous(), w, false);
  } else if (many_rows_win(M, N, K, false)) {
    return many_rows(x.contiguous(), w, false);
  }
  // Cold weights: W streamed once past up to 256 rows wins for 4096 to 8192 outputs above 128
  // rows (6144 x 4096 1.36 and 1.18 TB/s), and up to there for long K and more outputs than
  // the kernel above takes. AURORA_SKINNY3=0 leaves them to the library.
  if (M > 64 && M <= 256 && N % 64 == 0 &&
      (M <= 128 ? K >= 8192 : N > 4096 && N <= 8192 && K <= 4096)) {
    const char* off = std::getenv("AURORA_SKINNY3");
    if (!off || std::strcmp(off, "0")) return skinny_gemm3_ex(x.contiguous(), w, 384);
  }
  return {};
}
