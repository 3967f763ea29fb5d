// The large-tile wide GEMM (gemm16t.h) for Q5_K, Q6_K and Q8_0 weights.
#include "gemm16t.h"

namespace {

template <class F, int EPI>
void dispatch(sh_engine* e, const QMat& w, const uint16_t* bh, uint32_t ldb, uint32_t N, const Gemm16tPlan& p,
              const EpiArgs& ea) {
  constexpr int kMost = (F::kStage > 2048) ? 6 : 8;  // Q8_0: the stages of 8 groups exceed the LDS
  if (p.CG == 4) launch<F, 4, EPI>(e, w, bh, ldb, N, p, ea);
  else if (p.CG == 6) launch<F, 6, EPI>(e, w, bh, ldb, N, p, ea);
  else launch<F, kMost, EPI>(e, w, bh, ldb, N, p, ea);
}

template <class F>
void dispatch_epi(sh_engine* e, const QMat& w, const uint16_t* bh, uint32_t ldb, uint32_t N, const Gemm16tPlan& p,
                  EpiKind epi, const EpiArgs& ea) {
  switch (epi) {
    case EPI_PART: dispatch<F, EPI_PART>(e, w, bh, ldb, N, p, ea); break;
    case EPI_ADD: dispatch<F, EPI_ADD>(e, w, bh, ldb, N, p, ea); break;
    case EPI_QKV: dispatch<F, EPI_QKV>(e, w, bh, ldb, N, p, ea); break;
    case EPI_SWIGLU: dispatch<F, EPI_SWIGLU>(e, w, bh, ldb, N, p, ea); break;
    default: dispatch<F, EPI_STORE>(e, w, bh, ldb, N, p, ea); break;
  }
}

}  // namespace

void sh_gemm16t_fmt_launch(sh_engine* e, const QMat& w, const uint16_t* bh, uint32_t ldb, uint32_t N,
                           const Gemm16tPlan& p, EpiKind epi, const EpiArgs& ea) {
  if (w.type == GGML_Q8_0) dispatch_epi<Q8>(e, w, bh, ldb, N, p, epi, ea);
  else if (w.type == GGML_Q5_K) dispatch_epi<Q5K>(e, w, bh, ldb, N, p, epi, ea);
  else dispatch_epi<Q6K>(e, w, bh, ldb, N, p, epi, ea);
}
