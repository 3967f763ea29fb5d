// The large-tile wide GEMM (gemm16t.h): split plans and the Q4_K launches.
#include <algorithm>

#include "gemm16t.h"

namespace {

template <class F, int EPI>
void dispatch(sh_engine* e, const QMat& w, const uint16_t* bh, uint32_t ldb, uint32_t N, const Gemm16tPlan& p,
              const EpiArgs& ea) {
  switch (p.CG) {
    case 3: launch<F, 3, EPI>(e, w, bh, ldb, N, p, ea); break;
    case 4: launch<F, 4, EPI>(e, w, bh, ldb, N, p, ea); break;
    case 5: launch<F, 5, EPI>(e, w, bh, ldb, N, p, ea); break;
    case 6: launch<F, 6, EPI>(e, w, bh, ldb, N, p, ea); break;
    case 7: launch<F, 7, EPI>(e, w, bh, ldb, N, p, ea); break;
    default: launch<F, 8, EPI>(e, w, bh, ldb, N, p, ea); break;
  }
}

}  // namespace

// Whether the kernel takes w: whole stages of 128 k (K-quants: superblocks).
bool sh_gemm16t_ok(const QMat& w) {
  return sh_is_kquant(w.type) ? w.K % 256 == 0 : w.type == GGML_Q8_0 && w.K % 128 == 0;
}

// The split plan minimises an estimate of the call's time (us, fitted to the 8B
// shapes at 65 - 2048 columns): rounds of one workgroup per CU, each kHalf(CG)
// per 128 k plus the fill of the pipeline and the epilogue, plus, with several
// splits, the partials' write and their read at ~4 TB/s by the finishing launch
// that a single split does without.
Gemm16tPlan sh_gemm16t_plan(const QMat& w, bool one_split, uint32_t N) {
  const uint32_t unit = w.type == GGML_Q8_0 ? 1 : 2;  // stages a split boundary may fall between
  const uint32_t G = (N + 31) / 32, nu = w.K / 128 / unit, nrb = (w.tiles + 15) / 16, slots = 256;
  const bool q4 = w.type == GGML_Q4_K;
  const size_t col_bytes = (size_t)((N + 7) / 8 * 8) * w.tiles * 16 * 4;
  const uint32_t cap = one_split ? 1 : (uint32_t)std::max<size_t>(1, std::min<size_t>(16, SH_PART16_BYTES / col_bytes));
  Gemm16tPlan p;
  double best = 1e300;
  uint32_t last_ncb = 0;
  for (uint32_t cg = w.type == GGML_Q8_0 ? 6 : 8; cg >= 3; --cg) {
    const uint32_t ncb = (G + cg - 1) / cg;
    uint32_t even = std::max(3u, (G + ncb - 1) / ncb);
    if (!q4) even = (std::max(4u, even) + 1) / 2 * 2;  // the other formats come in 4, 6 and 8 groups
    if (ncb == last_ncb) continue;  // the same blocks, evened out already
    last_ncb = ncb;
    for (uint32_t ks = 1; ks <= cap && ks <= nu; ++ks) {
      const uint32_t S = (nu + ks - 1) / ks, k2 = (nu + S - 1) / S, wgs = nrb * ncb * k2;
      if (k2 != ks) continue;
      const double part_us = k2 > 1 ? (double)k2 * col_bytes * 2 / 4e6 + 2.0 : 0.0;
      const double cost = (double)((wgs + slots - 1) / slots) * (unit * S * (0.85 + 0.27 * even) + 8.0) + part_us;
      if (cost < best - 1e-9) {
        best = cost;
        p.CG = even; p.ncb = ncb; p.HS = unit * S; p.KS = k2;
      }
    }
  }
  return p;
}

int sh_gemm16t_launch(sh_engine* e, const QMat& w, const uint16_t* bh, uint32_t ldb, uint32_t N, const Gemm16tPlan& p,
                      EpiKind epi, const EpiArgs& ea) {
  SH_CHECK(sh_gemm16t_ok(w) && ldb >= w.K && ldb % 8 == 0 && N >= 1 && N <= 32 * p.CG * p.ncb &&
               (uint64_t)N * ldb * 2 < (1ull << 32),
           SH_ERR_ARG, "f16 gemm: type %d, K %u, ldb %u, N %u", w.type, w.K, ldb, N);
  SH_CHECK(epi == EPI_PART || p.KS == 1, SH_ERR_ARG, "f16 gemm: epilogue %d needs whole sums", (int)epi);
  SH_CHECK(epi != EPI_QKV || (ea.tab && ea.out && ea.hd % 4 == 0 && ea.row_base % 4 == 0 && ea.Dq % 64 == 0 &&
                              ea.Dkv % 64 == 0 && ea.row_base + w.M <= ea.Dq + 2 * ea.Dkv),
           SH_ERR_ARG, "f16 gemm: QKV epilogue shape");
  SH_CHECK(epi != EPI_SWIGLU || (ea.h16 && w.tiles % 2 == 0 && ea.ldh % 4 == 0 && ea.ldh >= w.tiles * 8), SH_ERR_ARG,
           "f16 gemm: SwiGLU epilogue shape");
  if (w.type != GGML_Q4_K) sh_gemm16t_fmt_launch(e, w, bh, ldb, N, p, epi, ea);
  else if (epi == EPI_PART) dispatch<Q4K, EPI_PART>(e, w, bh, ldb, N, p, ea);
  else if (epi == EPI_ADD) dispatch<Q4K, EPI_ADD>(e, w, bh, ldb, N, p, ea);
  else if (epi == EPI_QKV) dispatch<Q4K, EPI_QKV>(e, w, bh, ldb, N, p, ea);
  else if (epi == EPI_SWIGLU) dispatch<Q4K, EPI_SWIGLU>(e, w, bh, ldb, N, p, ea);
  else dispatch<Q4K, EPI_STORE>(e, w, bh, ldb, N, p, ea);
  SH_HIP(hipGetLastError());
  return SH_OK;
}
