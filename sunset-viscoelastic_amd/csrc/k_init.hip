// k_init.hip -- the initial state of the time loop, made on the device from the
// caller's arrays: state records (rou = ro u, psi = log c in the
// log-conformation form), the Kolmogorov forcing and the sum of the node
// volumes.  (On the host, with the node arrays copied back and forth and two
// logarithms a node, this was most of sv_set_initial: 11 ms of 262k nodes,
// and 0.3 ms of every sv_set_phys on 16k.)
#include "sv_internal.h"

namespace {

constexpr int IB = 256;

// log_conf_psi_from_c (conf_transforms.F90:177-215); uncontracted, so that the
// cancellations of its nearly isotropic branch fall as they do on the host
__device__ __forceinline__ void psi_from_c(double a, double b, double d, double &pxx, double &pxy,
                                           double &pyy) {
#pragma clang fp contract(off)
  double l1, l2, R[4];
  if (fabs(b) <= 1.0e-16) {
    l1 = a; l2 = d; R[0] = 1; R[1] = 0; R[2] = 0; R[3] = 1;
  } else {
    const double tr = a + d, det = a * d - b * b;
    double t = 0.25 * tr * tr - det;
    if (t <= 1.0e-16) t = 0.0;
    t = sqrt(t);
    l1 = 0.5 * tr + t;
    l2 = 0.5 * tr - t;
    double r11 = l1 - d, r21 = b;
    const double nrm = sqrt(r11 * r11 + r21 * r21);
    r11 /= nrm; r21 /= nrm;
    R[0] = r11; R[1] = r21; R[2] = -r21; R[3] = r11;
  }
  const double e1 = log(l1), e2 = log(l2);
  const double i11 = e1 * R[0], i12 = e1 * R[1], i21 = e2 * R[2], i22 = e2 * R[3];
  pxx = R[0] * i11 + R[2] * i21;
  pxy = R[1] * i11 + R[3] * i21;
  pyy = R[1] * i12 + R[3] * i22;
}

// record k holds the caller's node perm[k]; f: ro, u, v, cxx, cxy, cyy
__global__ __launch_bounds__(IB) void k_init_records(int n, const int *perm, const double *f,
                                                     int lc, double *U) {
  const int k = blockIdx.x * IB + threadIdx.x;
  if (k >= n) return;
  const int i = perm[k];
  const size_t N = n;
  const double ro = f[i];
  double r[6] = {ro, ro * f[N + i], ro * f[2 * N + i], f[3 * N + i], f[4 * N + i], f[5 * N + i]};
  if (lc) psi_from_c(r[3], r[4], r[5], r[3], r[4], r[5]);
  double2 *u = reinterpret_cast<double2 *>(U + (size_t)SV_US * k);
  u[0] = double2{r[0], r[1]};
  u[1] = double2{r[2], r[3]};
  u[2] = double2{r[4], r[5]};
}

__global__ __launch_bounds__(IB) void k_forcing(int n, const int *perm, const double *y,
                                                double amp, double wave, double *fx) {
  const int k = blockIdx.x * IB + threadIdx.x;
  if (k < n) fx[k] = amp * sin(wave * y[perm[k]]);
}

// one block: a fixed-order sum of n values
__global__ __launch_bounds__(1024) void k_total(int n, const double *v, double *out) {
  __shared__ double s[1024];
  double a = 0.0;
#pragma unroll 4
  for (int k = threadIdx.x; k < n; k += 1024) a += v[k];
  s[threadIdx.x] = a;
  __syncthreads();
  for (int o = 512; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) s[threadIdx.x] += s[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = s[0];
}

// (two copies of the block across the bus, each waited for, cost 30 us)
__global__ void k_set_control(sv_ctrl *c, double dt, double time, int itime, double e1, double e2,
                              double e3, int dt_mode) {
  c->dt = dt; c->time = time; c->itime = itime;
  c->emax_np1 = e1; c->emax_n = e2; c->emax_nm1 = e3;
  c->dt_mode = dt_mode;
}

}  // namespace

int sv_dev_set_control(sv_ctx *c, double dt, double time, int itime, double e1, double e2,
                       double e3, int dt_mode) {
  k_set_control<<<1, 1, 0, c->stream>>>(c->ctrl, dt, time, itime, e1, e2, e3, dt_mode);
  SV_HIP(c, hipGetLastError());
  SV_HIP(c, hipStreamSynchronize(c->stream));   // diagnostics read it on other streams
  return 0;
}

int sv_dev_init_records(sv_ctx *c, const double *fields) {
  const int n = c->npfb;
  k_init_records<<<(n + IB - 1) / IB, IB, 0, c->stream>>>(n, c->L.perm, fields,
                                                          c->cfg.form == SV_FORM_LC, c->U);
  SV_HIP(c, hipGetLastError());
  return 0;
}

int sv_dev_forcing(sv_ctx *c) {
  const int n = c->npfb;
  k_forcing<<<(n + IB - 1) / IB, IB, 0, c->stream>>>(n, c->L.perm, c->y, c->pk.kol_amp,
                                                     c->pk.kol_k, c->fx);
  SV_HIP(c, hipGetLastError());
  return 0;
}

int sv_dev_volume_sum(sv_ctx *c, double *sum) {
  // a scratch value past the partial results
  double *out = c->partial + c->npartial;
  k_total<<<1, 1024, 0, c->stream>>>(c->npfb, c->vol, out);
  SV_HIP(c, hipGetLastError());
  SV_HIP(c, hipMemcpyAsync(sum, out, sizeof(double), hipMemcpyDeviceToHost, c->stream));
  SV_HIP(c, hipStreamSynchronize(c->stream));
  return 0;
}
