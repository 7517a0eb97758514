// One unit of the register-transform edges: instantiates the z, y and x passes of the lengths
// QBH_EDGES_<QBH_FFT_PART> lists, in FP64 (E and D) and FP32 (E and F).
#include "qbh_fft_edges.h"
#include "qbh_fft_kernels.h"

#define QBH_CAT_(a, b) a##b
#define QBH_CAT(a, b) QBH_CAT_(a, b)
#define QBH_EDGE64(N1, N2) make_edge<double, N1, N2>(),
#define QBH_EDGE32(N1, N2) make_edge<float, N1, N2>(),
#define QBH_NO_EDGE(N1, N2)

namespace qbh {

static const EdgeOps kOps64[] = {QBH_CAT(QBH_EDGES_, QBH_FFT_PART)(QBH_EDGE64, QBH_EDGE64, QBH_NO_EDGE)};
static const EdgeOps kOps32[] = {QBH_CAT(QBH_EDGES_, QBH_FFT_PART)(QBH_EDGE32, QBH_NO_EDGE, QBH_EDGE32)};

EdgeTable QBH_CAT(edge_table_, QBH_FFT_PART)(int prec) {
  if (prec == PREC_FP64) return {kOps64, (int)(sizeof(kOps64) / sizeof(kOps64[0]))};
  return {kOps32, (int)(sizeof(kOps32) / sizeof(kOps32[0]))};
}

}  // namespace qbh
