// Layers of one 2x2 gate on every qubit (U^(x)n), forward and adjoint: the QAOA mixer
// exp(-i beta sum_q X_q) = prod_q RX_q(2 beta) and its backward step.  Entry points in
// include/iqs_hip.h ("layers"); kernels in iqs_layer.hpp.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>

#include "../../include/iqs_hip.h"
#include "iqs_layer.hpp"

using namespace iqsl;

namespace {

struct LayerWork {
  double* part = nullptr;
  size_t have = 0;
  double* host = nullptr;  // pinned: the sums are written here by the kernel
  size_t host_have = 0;
};
LayerWork g_lw;
std::mutex g_lm;  // one layer call at a time uses g_lw, until its sums are on the host
// Partials kept on the device before they are summed (32 MiB), unless one group needs more.
constexpr uint64_t kPartCap = uint64_t(1) << 22;

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

int layer(const LayerArgs& a, LayerShape* shape = nullptr)
{
  return a.psi->dtype == IQSH_C128 ? do_layer<double>(a, shape) : do_layer<float>(a, shape);
}

// One backward step, results summed into *dmixer (and *dgamma with a phase).
int adjoint_once(LayerArgs a, double* dmixer, double* dgamma)
{
  LayerShape sh;
  if (int rc = layer(a, &sh)) return rc;
  const int group = (int)sh.passes + (a.cs ? 1 : 0);
  LayerSums sums;
  if (int rc = sums.begin(sh.run, 2, group)) return rc;
  a.sums = &sums;
  if (int rc = layer(a)) return rc;
  const double* r;
  if (int rc = sums.finish(&r)) return rc;
  double s = 0;
  for (unsigned i = 0; i < sh.passes; ++i) s += r[i];
  *dmixer = 2.0 * s;
  if (a.cs) *dgamma = 2.0 * r[sh.passes];
  return IQSH_OK;
}

// RX(2 beta), the mixer of one layer (and of its inverse for -beta).
void mixer_of(double beta, double m[8])
{
  const double theta = 2.0 * beta, c = std::cos(theta / 2.0), s = std::sin(theta / 2.0);
  const double r[8] = {c, 0, 0, -s, 0, -s, c, 0};
  std::copy(r, r + 8, m);
}

const double kGenX[8] = {0, 0, 1, 0, 1, 0, 0, 0};

}  // namespace

namespace iqsl {

int LayerSums::begin(uint64_t run, int group, uint64_t total)
{
  if (g_lw.host_have < total) {
    IQSI_TRY(hipStreamSynchronize(iqsi::stream()));
    if (g_lw.host) IQSI_TRY(hipHostFree(g_lw.host));
    g_lw.host = nullptr;
    g_lw.host_have = 0;
    const size_t want = std::max<size_t>(total, 512);
    IQSI_TRY(hipHostMalloc((void**)&g_lw.host, sizeof(double) * want, hipHostMallocDefault));
    g_lw.host_have = want;
  }
  const uint64_t count = std::max<uint64_t>(std::min<uint64_t>(run * total, kPartCap), run * group);
  if (g_lw.have < count) {
    IQSI_TRY(hipStreamSynchronize(iqsi::stream()));
    if (g_lw.part) IQSI_TRY(hipFree(g_lw.part));
    g_lw.part = nullptr;
    g_lw.have = 0;
    if (hipMalloc((void**)&g_lw.part, sizeof(double) * count) != hipSuccess)
      return iqsi::fail(IQSH_ERR_ALLOC, "layer reduction buffer of %zu doubles", (size_t)count);
    g_lw.have = count;
  }
  return IQSH_OK;
}

int LayerSums::take(uint64_t run, int count, double** part)
{
  if (n_ + count > kMaxSums || used_ + run * count > g_lw.have)
    if (int rc = flush()) return rc;
  if (run * count > g_lw.have || taken() + count > g_lw.host_have)
    return iqsi::fail(IQSH_ERR_ARG, "layer sums beyond the space reserved for them");
  *part = g_lw.part + used_;
  for (int i = 0; i < count; ++i) {
    runs_.off[n_] = used_;
    runs_.len[n_++] = run;
    used_ += run;
  }
  return IQSH_OK;
}

int LayerSums::flush()
{
  if (!n_) return IQSH_OK;
  k_sum_runs<<<n_, kSumB, 0, iqsi::stream()>>>(g_lw.part, runs_, g_lw.host + done_);
  IQSI_TRY(hipGetLastError());
  done_ += n_;
  n_ = 0;
  used_ = 0;
  return IQSH_OK;
}

int LayerSums::finish(const double** results)
{
  if (int rc = flush()) return rc;
  IQSI_TRY(hipStreamSynchronize(iqsi::stream()));
  *results = g_lw.host;
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
  return layer({h, nullptr, m, nullptr, nullptr, nullptr});
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
  return layer({h, nullptr, mixer, nullptr, &cs, nullptr});
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
  return adjoint_once({psi, lam, mixer_inv, G, &cs, nullptr}, dmixer, dgamma);
}

int iqsh_adjoint_1q_all(iqsh_handle psi, iqsh_handle lam, const double Uinv[8], const double* G, double* grad)
{
  if (int rc = check_adjoint(psi, lam)) return rc;
  if (!Uinv || !G || !grad) return iqsi::fail(IQSH_ERR_ARG, "null argument");
  if (int rc = check_size(psi)) return rc;
  std::lock_guard<std::mutex> lk(g_lm);
  return adjoint_once({psi, lam, Uinv, G, nullptr, nullptr}, grad, nullptr);
}

int iqsh_qaoa_run(iqsh_handle psi, unsigned layers, unsigned ne, const unsigned* u, const unsigned* v, const double* w,
                  const double* gammas, const double* betas)
{
  if (int rc = check_layer(psi)) return rc;
  if ((layers && (!gammas || !betas)) || (ne && (!u || !v))) return iqsi::fail(IQSH_ERR_ARG, "null argument");
  if (int rc = check_size(psi)) return rc;
  CutSpec cs;
  if (int rc = iqsi::build_cut_spec(psi, ne, u, v, w, 0.0, &cs)) return rc;  // the edges are in order
  if (int rc = iqsh_init_uniform(psi, 1.0 / std::sqrt((double)psi->size()), 0.0)) return rc;
  std::lock_guard<std::mutex> lk(g_lm);
  for (unsigned l = 0; l < layers; ++l) {
    double m[8];
    mixer_of(betas[l], m);
    if (int rc = iqsi::build_cut_spec(psi, ne, u, v, w, gammas[l], &cs)) return rc;
    if (int rc = layer({psi, nullptr, m, nullptr, &cs, nullptr})) return rc;
  }
  return IQSH_OK;
}

int iqsh_qaoa_gradient(iqsh_handle psi, iqsh_handle lam, unsigned layers, unsigned ne, const unsigned* u,
                       const unsigned* v, const double* w, const double* gammas, const double* betas, double* cost,
                       double* dgammas, double* dbetas)
{
  if (int rc = check_adjoint(psi, lam)) return rc;
  if (!cost || (layers && (!gammas || !betas || !dgammas || !dbetas)) || (ne && (!u || !v)))
    return iqsi::fail(IQSH_ERR_ARG, "null argument");
  if (int rc = check_size(psi)) return rc;
  CutSpec cs;
  if (int rc = iqsi::build_cut_spec(psi, ne, u, v, w, 0.0, &cs)) return rc;
  std::lock_guard<std::mutex> lk(g_lm);
  LayerArgs a{psi, lam, nullptr, kGenX, &cs, nullptr};
  const double one[8] = {1, 0, 0, 0, 0, 0, 1, 0};
  a.u = one;
  LayerShape sh;
  if (int rc = layer(a, &sh)) return rc;
  const uint64_t per = sh.passes + 1;
  const unsigned nc = iqsi::cost_blocks(psi);
  LayerSums sums;
  if (int rc = sums.begin(std::max<uint64_t>(sh.run, nc), 2, 1 + per * layers)) return rc;
  a.sums = &sums;
  double* part;
  if (int rc = sums.take(nc, 1, &part)) return rc;
  if (int rc = iqsi::launch_cost(psi, lam, cs, part)) return rc;
  for (unsigned i = 0; i < layers; ++i) {
    const unsigned l = layers - 1 - i;
    double m[8];
    mixer_of(-betas[l], m);
    // Un-applying exp(-i gamma C) is applying exp(-i (-gamma) C).
    if (int rc = iqsi::build_cut_spec(psi, ne, u, v, w, -gammas[l], &cs)) return rc;
    a.u = m;
    if (int rc = layer(a)) return rc;
  }
  const double* r;
  if (int rc = sums.finish(&r)) return rc;
  *cost = r[0];
  for (unsigned i = 0; i < layers; ++i) {
    const double* x = r + 1 + per * i;
    double s = 0;
    for (unsigned k = 0; k < sh.passes; ++k) s += x[k];
    dbetas[layers - 1 - i] = 2.0 * s;
    dgammas[layers - 1 - i] = 2.0 * x[sh.passes];
  }
  return IQSH_OK;
}

}  // extern "C"
