// Layers of one 2x2 gate on every qubit (U^(x)n), forward and adjoint: the QAOA mixer
// exp(-i beta sum_q X_q) = prod_q RX_q(2 beta) and its backward step.  Entry points in
// include/iqs_hip.h ("layers"); kernels in iqs_layer.hpp.
#include <hip/hip_runtime.h>

#include <mutex>

#include "../../include/iqs_hip.h"
#include "iqs_layer.hpp"

using namespace iqsl;

namespace {

struct LayerWork {
  double* part = nullptr;
  size_t have = 0;
  double* host = nullptr;  // pinned: the sums are written here by the kernel
};
LayerWork g_lw;
std::mutex g_lm;  // one layer call at a time uses g_lw, until its sums are on the host

constexpr int kSumB = 1024;

// out[i] = sum of run i's partials in a fixed order, one workgroup per run: thread t adds
// part[t], part[t + kSumB], ... in eight interleaved chains (so that eight loads are in
// flight), then the workgroup sum.
__global__ __launch_bounds__(kSumB) void k_sum_runs(const double* __restrict__ part, SumRuns runs, double* __restrict__ out)
{
  const double* p = part + runs.off[blockIdx.x];
  const uint64_t n = runs.len[blockIdx.x];
  double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  uint64_t i = threadIdx.x;
  for (; i + 7 * kSumB < n; i += 8 * kSumB)
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] += p[i + u * kSumB];
  for (; i < n; i += kSumB) v[0] += p[i];
  wg_sum_store<kSumB>(((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])), out + blockIdx.x);
}

// The layer kernels need a tile of 2^10 amplitudes.
constexpr unsigned kMinLayerQubits = 10;

int check_layer(iqsh_handle h)
{
  if (!h || !h->d) return iqsi::fail(IQSH_ERR_ARG, "null or released state handle");
  return IQSH_OK;
}

int check_adjoint(iqsh_handle psi, iqsh_handle lam)
{
  if (int rc = check_layer(psi)) return rc;
  if (int rc = check_layer(lam)) return rc;
  if (psi->n != lam->n || psi->dtype != lam->dtype) return iqsi::fail(IQSH_ERR_ARG, "registers differ in size or precision");
  return IQSH_OK;
}

int check_size(iqsh_handle h)
{
  if (h->n < kMinLayerQubits) return iqsi::fail(IQSH_ERR_NOTSUP, "layer kernels need >= %u qubits", kMinLayerQubits);
  return IQSH_OK;
}

int layer(const LayerArgs& a) { return a.psi->dtype == IQSH_C128 ? do_layer<double>(a) : do_layer<float>(a); }

}  // namespace

namespace iqsl {

int layer_parts(uint64_t count, double** part)
{
  if (!g_lw.host) IQSI_TRY(hipHostMalloc((void**)&g_lw.host, sizeof(double) * kMaxSums, hipHostMallocDefault));
  if (g_lw.have < count) {
    IQSI_TRY(hipStreamSynchronize(iqsi::stream()));
    if (g_lw.part) IQSI_TRY(hipFree(g_lw.part));
    g_lw.part = nullptr;
    g_lw.have = 0;
    if (hipMalloc((void**)&g_lw.part, sizeof(double) * count) != hipSuccess)
      return iqsi::fail(IQSH_ERR_ALLOC, "layer reduction buffer of %zu doubles", (size_t)count);
    g_lw.have = count;
  }
  *part = g_lw.part;
  return IQSH_OK;
}

int layer_sums(const SumRuns& runs, int nsum, double* out)
{
  k_sum_runs<<<nsum, kSumB, 0, iqsi::stream()>>>(g_lw.part, runs, g_lw.host);
  IQSI_TRY(hipGetLastError());
  IQSI_TRY(hipStreamSynchronize(iqsi::stream()));
  for (int i = 0; i < nsum; ++i) out[i] = g_lw.host[i];
  return IQSH_OK;
}

}  // namespace iqsl

extern "C" {

int iqsh_apply_1q_all(iqsh_handle h, const double m[8])
{
  if (int rc = check_layer(h)) return rc;
  if (!m) return iqsi::fail(IQSH_ERR_ARG, "null matrix");
  if (int rc = check_size(h)) return rc;
  std::lock_guard<std::mutex> lk(g_lm);
  return layer({h, nullptr, m, nullptr, nullptr, nullptr, nullptr});
}

int iqsh_qaoa_layer(iqsh_handle h, unsigned ne, const unsigned* u, const unsigned* v, const double* w, double gamma,
                    const double mixer[8])
{
  if (int rc = check_layer(h)) return rc;
  if (!mixer || (ne && (!u || !v))) return iqsi::fail(IQSH_ERR_ARG, "null argument");
  if (int rc = check_size(h)) return rc;
  CutSpec cs;
  if (int rc = iqsi::build_cut_spec(h, ne, u, v, w, gamma, &cs)) return rc;
  std::lock_guard<std::mutex> lk(g_lm);
  return layer({h, nullptr, mixer, nullptr, &cs, nullptr, nullptr});
}

int iqsh_qaoa_layer_adjoint(iqsh_handle psi, iqsh_handle lam, unsigned ne, const unsigned* u, const unsigned* v,
                            const double* w, double gamma, const double mixer_inv[8], const double* G,
                            double* dgamma, double* dmixer)
{
  if (int rc = check_adjoint(psi, lam)) return rc;
  if (!mixer_inv || !G || !dgamma || !dmixer || (ne && (!u || !v))) return iqsi::fail(IQSH_ERR_ARG, "null argument");
  if (int rc = check_size(psi)) return rc;
  CutSpec cs;
  // Un-applying exp(-i gamma C) is applying exp(-i (-gamma) C).
  if (int rc = iqsi::build_cut_spec(psi, ne, u, v, w, -gamma, &cs)) return rc;
  std::lock_guard<std::mutex> lk(g_lm);
  return layer({psi, lam, mixer_inv, G, &cs, dmixer, dgamma});
}

int iqsh_adjoint_1q_all(iqsh_handle psi, iqsh_handle lam, const double Uinv[8], const double* G, double* grad)
{
  if (int rc = check_adjoint(psi, lam)) return rc;
  if (!Uinv || !G || !grad) return iqsi::fail(IQSH_ERR_ARG, "null argument");
  if (int rc = check_size(psi)) return rc;
  std::lock_guard<std::mutex> lk(g_lm);
  return layer({psi, lam, Uinv, G, nullptr, grad, nullptr});
}

}  // extern "C"
