// The any-lattice ResConv kernels (resconv_wave.hpp): 32 channels, FP32.
// Classes (waves per configuration, tiles per wave, least tiles of a wave)
// follow rw_pick.
#include "resconv_wave.hpp"

namespace qtx {

template <>
int rw_logpsi<32, QTX_CONV_FP32>(hipStream_t st, const RcLayout& L, const RcArgs& a, const int8_t* s, int64_t ns,
                                double* logabs) {
  const RwPick pk = rw_pick(32, L.N, ns);
  if (pk.P == 1 && pk.maxt == 4) {
    RW_LAUNCH(rw_logpsi_kernel, 32, QTX_CONV_FP32, 4, 1, 1, 0, (ns + G - 1) / G,
              s, ns, logabs);
    QTX_LAUNCH_CHECK();
    return QTX_OK;
  }
  if (pk.P == 2 && pk.maxt == 4) {
    RW_LAUNCH(rw_logpsi_kernel, 32, QTX_CONV_FP32, 4, 2, 2, 0, (ns + G - 1) / G,
              s, ns, logabs);
    QTX_LAUNCH_CHECK();
    return QTX_OK;
  }
  if (pk.P == 4 && pk.maxt == 2) {
    RW_LAUNCH(rw_logpsi_kernel, 32, QTX_CONV_FP32, 2, 4, 0, 0, (ns + G - 1) / G,
              s, ns, logabs);
    QTX_LAUNCH_CHECK();
    return QTX_OK;
  }
  if (pk.P == 4 && pk.maxt == 4) {
    RW_LAUNCH(rw_logpsi_kernel, 32, QTX_CONV_FP32, 4, 4, 2, 0, (ns + G - 1) / G,
              s, ns, logabs);
    QTX_LAUNCH_CHECK();
    return QTX_OK;
  }
  if (pk.P == 4 && pk.maxt == 7) {
    RW_LAUNCH(rw_logpsi_kernel, 32, QTX_CONV_FP32, 7, 4, 4, 0, (ns + G - 1) / G,
              s, ns, logabs);
    QTX_LAUNCH_CHECK();
    return QTX_OK;
  }
  return fail(QTX_EINVAL, "no ResConv kernel of this size class");
}

template <>
int rw_metropolis<32, QTX_CONV_FP32>(hipStream_t st, const RcLayout& L, const RcArgs& a, int kind, const int32_t* nbr,
                                    int width, int hopping, const uint32_t* words, int nsteps, int64_t ns,
                                    double reweight, double tie_tol, int8_t* s, double* logabs, int32_t* n_accept,
                                    int32_t* n_near) {
  const RwPick pk = rw_pick(32, L.N, ns, true);
  if (pk.P == 1 && pk.maxt == 4) {
    RW_LAUNCH(rw_metropolis_kernel, 32, QTX_CONV_FP32, 4, 1, 1, 0, (ns + G - 1) / G,
              kind, nbr, width, hopping, words, nsteps, ns, reweight, tie_tol, s, logabs, n_accept, n_near);
    QTX_LAUNCH_CHECK();
    return QTX_OK;
  }
  if (pk.P == 2 && pk.maxt == 4) {
    RW_LAUNCH(rw_metropolis_kernel, 32, QTX_CONV_FP32, 4, 2, 2, 0, (ns + G - 1) / G,
              kind, nbr, width, hopping, words, nsteps, ns, reweight, tie_tol, s, logabs, n_accept, n_near);
    QTX_LAUNCH_CHECK();
    return QTX_OK;
  }
  if (pk.P == 4 && pk.maxt == 2) {
    RW_LAUNCH(rw_metropolis_kernel, 32, QTX_CONV_FP32, 2, 4, 0, 0, (ns + G - 1) / G,
              kind, nbr, width, hopping, words, nsteps, ns, reweight, tie_tol, s, logabs, n_accept, n_near);
    QTX_LAUNCH_CHECK();
    return QTX_OK;
  }
  if (pk.P == 4 && pk.maxt == 4) {
    RW_LAUNCH(rw_metropolis_kernel, 32, QTX_CONV_FP32, 4, 4, 2, 0, (ns + G - 1) / G,
              kind, nbr, width, hopping, words, nsteps, ns, reweight, tie_tol, s, logabs, n_accept, n_near);
    QTX_LAUNCH_CHECK();
    return QTX_OK;
  }
  if (pk.P == 4 && pk.maxt == 7) {
    RW_LAUNCH(rw_metropolis_kernel, 32, QTX_CONV_FP32, 7, 4, 4, 0, (ns + G - 1) / G,
              kind, nbr, width, hopping, words, nsteps, ns, reweight, tie_tol, s, logabs, n_accept, n_near);
    QTX_LAUNCH_CHECK();
    return QTX_OK;
  }
  return fail(QTX_EINVAL, "no ResConv kernel of this size class");
}

template <>
int rw_eloc<32, QTX_CONV_FP32>(hipStream_t st, const RcLayout& L, const RcArgs& a, const qtx_ham& H, const int8_t* s,
                              const double* logabs, int64_t ns, int S, double* eloc, int32_t* nconn) {
  const RwPick pk = rw_eloc_pick(32, L.N, H.noff, ns);
  if (pk.P == 1 && pk.maxt == 4) {
    RW_LAUNCH(rw_eloc_kernel, 32, QTX_CONV_FP32, 4, 1, 1, H.noff, ns * S,
              H, s, logabs, S, eloc, nconn);
    QTX_LAUNCH_CHECK();
    return QTX_OK;
  }
  if (pk.P == 2 && pk.maxt == 4) {
    RW_LAUNCH(rw_eloc_kernel, 32, QTX_CONV_FP32, 4, 2, 2, H.noff, ns * S,
              H, s, logabs, S, eloc, nconn);
    QTX_LAUNCH_CHECK();
    return QTX_OK;
  }
  if (pk.P == 4 && pk.maxt == 2) {
    RW_LAUNCH(rw_eloc_kernel, 32, QTX_CONV_FP32, 2, 4, 0, H.noff, ns * S,
              H, s, logabs, S, eloc, nconn);
    QTX_LAUNCH_CHECK();
    return QTX_OK;
  }
  if (pk.P == 4 && pk.maxt == 4) {
    RW_LAUNCH(rw_eloc_kernel, 32, QTX_CONV_FP32, 4, 4, 2, H.noff, ns * S,
              H, s, logabs, S, eloc, nconn);
    QTX_LAUNCH_CHECK();
    return QTX_OK;
  }
  if (pk.P == 4 && pk.maxt == 7) {
    RW_LAUNCH(rw_eloc_kernel, 32, QTX_CONV_FP32, 7, 4, 4, H.noff, ns * S,
              H, s, logabs, S, eloc, nconn);
    QTX_LAUNCH_CHECK();
    return QTX_OK;
  }
  return fail(QTX_EINVAL, "no ResConv kernel of this size class");
}

}  // namespace qtx
