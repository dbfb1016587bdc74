// Device-resident particle state and j prediction (include/abyss_regf.h,
// abyss_ctx_upload_state / abyss_ctx_update_state / abyss_ctx_predict).
//
// The reference caller predicts every particle on the host, packs the
// arrays and copies all N of them before each regular step
// (src_mpi/cuda/CalculateRegularAcceleration.cpp:330-449, predictor
// src_mpi/Particle/UpdateParticle.cpp:37-59).  Here the state lives in HBM:
// the full state is uploaded once, after each corrector only the changed
// particles are scattered in, and a kernel predicts all j to the new time
// straight into the j-set the force kernels read.  The predictor evaluates
// the reference's expressions in the same order with FMA contraction off,
// so the predicted j-set is bitwise identical to a host prediction with
// plain IEEE double arithmetic.
#include "regf_context.h"

#include <stdio.h>
#include <string.h>

#include <cmath>

#include <algorithm>

namespace {

// State SoA (stride n): x[3][n], v[3][n], a[3][n], ad[3][n], t[n], m[n],
// r2[n] (all FP64).  Component-major so each kernel access is coalesced.
constexpr int kStateDoubles = 15;

struct StateView {
    const double *x, *v, *a, *ad, *t, *m, *r2;
};

StateView state_view(const double *base, int n)
{
    const size_t N = (size_t)n;
    return StateView{base, base + 3 * N, base + 6 * N, base + 9 * N, base + 12 * N, base + 13 * N,
                     base + 14 * N};
}

#pragma clang fp contract(off)
__global__ __launch_bounds__(256) void predict_kernel(StateView st, int n, double t_new,
                                                      double *__restrict__ jx,
                                                      float *__restrict__ m32,
                                                      abyss::JRec *__restrict__ aos)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t N = (size_t)n;
    const double h = t_new - st.t[i];
    double p[6];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const double x = st.x[d * N + i], v = st.v[d * N + i];
        double xp, vp;
        if (h == 0) {
            xp = x;
            vp = v;
        } else {
            const double a0 = st.a[d * N + i], a1 = st.ad[d * N + i];
            xp = ((a1 * h / 3 + a0) * h / 2 + v) * h + x;
            vp = (a1 * h / 2 + a0) * h + v;
        }
        jx[d * N + i] = xp;
        jx[(3 + d) * N + i] = vp;
        p[d] = xp;
        p[3 + d] = vp;
    }
    const double m = st.m[i];
    jx[6 * N + i] = m;
    jx[7 * N + i] = st.r2[i];
    m32[i] = (float)m;
    if (aos) aos[i] = abyss::JRec{p[0], p[1], p[2], p[3], p[4], p[5], m, 0.0};
}
#pragma clang fp contract(on)

// Scatter `count` updated particles (AoS records: x3 v3 a3 ad3 t m r2, read
// once from mapped host memory) into the SoA state.  A workgroup brings its
// records in as one run, by way of LDS.  Bound by the link's latency, from
// some 1000 records on by its rate and the host's packing; an update (1 / 513
// / 4096 / 16384 records) took 20.6 / 29.4 / 56 / 155 us with a copy to the
// device first, 18.8 / 22.6 / 47 / 141 in place.
__global__ __launch_bounds__(256) void scatter_kernel(double *__restrict__ state, int n,
                                                      const int *__restrict__ idx,
                                                      const double *__restrict__ rec, int count)
{
    constexpr int kRows = 64;
    __shared__ double s_rec[kRows * kStateDoubles];
    const int first = blockIdx.x * kRows;
    const int rows = min(kRows, count - first);
    const int k = threadIdx.x & (kRows - 1);
    const int i = k < rows ? idx[first + k] : 0;
    // every read over the link in flight at once
    constexpr int kLoads = (kRows * kStateDoubles + 255) / 256;
    double in[kLoads];
#pragma unroll
    for (int l = 0; l < kLoads; ++l) {
        const int e = min((int)threadIdx.x + 256 * l, rows * kStateDoubles - 1);
        in[l] = rec[(size_t)first * kStateDoubles + e];
    }
#pragma unroll
    for (int l = 0; l < kLoads; ++l) {
        const int e = threadIdx.x + 256 * l;
        if (e < rows * kStateDoubles) s_rec[e] = in[l];
    }
    __syncthreads();
    if (k >= rows) return;
    for (int c = threadIdx.x / kRows; c < kStateDoubles; c += 256 / kRows)
        state[(size_t)c * n + i] = s_rec[k * kStateDoubles + c];
}

}  // namespace

extern "C" {

int abyss_ctx_upload_state(abyss_ctx_t c, int n, const double *m, const double *x,
                           const double *v, const double *a, const double *adot, const double *t,
                           const double *r2)
{
    if (!c) return ABYSS_ERR_INVALID_ARG;
    if (n <= 0 || !m || !x || !v || !a || !adot || !t || !r2) {
        snprintf(c->detail, sizeof(c->detail), "upload_state: n=%d or null array", n);
        return ABYSS_ERR_INVALID_ARG;
    }
    for (int j = 0; j < n; ++j) {
        for (int d = 0; d < 3; ++d)
            if (!std::isfinite(x[3 * j + d]) || !std::isfinite(v[3 * j + d]) || !std::isfinite(a[3 * j + d]) ||
                !std::isfinite(adot[3 * j + d])) {
                snprintf(c->detail, sizeof(c->detail), "upload_state: non-finite data at j=%d", j);
                return ABYSS_ERR_INVALID_INPUT;
            }
        if (!std::isfinite(m[j]) || m[j] < 0.0 || !std::isfinite(t[j]) || std::isnan(r2[j]) || r2[j] < 0.0) {
            snprintf(c->detail, sizeof(c->detail), "upload_state: bad m/t/r2 at j=%d", j);
            return ABYSS_ERR_INVALID_INPUT;
        }
    }
    // an ordinary upload of the current positions sizes and fills the j-set
    int rc = abyss_ctx_upload(c, n, m, x, v, r2);
    if (rc != ABYSS_OK) return rc;
    const size_t bytes = (size_t)n * kStateDoubles * sizeof(double);
    if (hipSetDevice(c->device) != hipSuccess) return ABYSS_ERR_HIP;
    if (hipStreamSynchronize(c->stream) != hipSuccess) return ABYSS_ERR_HIP;
    if (bytes > c->state_bytes) {
        if (c->d_state) (void)hipFree(c->d_state);
        if (c->h_state) (void)hipHostFree(c->h_state);
        c->d_state = nullptr;
        c->h_state = nullptr;
        c->state_bytes = 0;
        if (hipMalloc(&c->d_state, bytes) != hipSuccess ||
            hipHostMalloc(&c->h_state, bytes, hipHostMallocDefault) != hipSuccess)
            return ABYSS_ERR_OUT_OF_MEMORY;
        c->state_bytes = bytes;
    }
    double *h = c->h_state;
    const size_t N = (size_t)n;
    for (int j = 0; j < n; ++j) {
        for (int d = 0; d < 3; ++d) {
            h[d * N + j] = x[3 * j + d];
            h[(3 + d) * N + j] = v[3 * j + d];
            h[(6 + d) * N + j] = a[3 * j + d];
            h[(9 + d) * N + j] = adot[3 * j + d];
        }
        h[12 * N + j] = t[j];
        h[13 * N + j] = m[j];
        h[14 * N + j] = r2[j];
    }
    if (hipMemcpyAsync(c->d_state, h, bytes, hipMemcpyHostToDevice, c->stream) != hipSuccess)
        return ABYSS_ERR_HIP;
    c->state_n = n;
    return ABYSS_OK;
}

int abyss_ctx_update_state(abyss_ctx_t c, int count, const int *idx, const double *m,
                           const double *x, const double *v, const double *a,
                           const double *adot, const double *t, const double *r2)
{
    if (!c) return ABYSS_ERR_INVALID_ARG;
    if (c->state_n <= 0) {
        snprintf(c->detail, sizeof(c->detail), "update_state before upload_state");
        return ABYSS_ERR_NO_JSET;
    }
    if (count <= 0 || !idx || !m || !x || !v || !a || !adot || !t || !r2) {
        snprintf(c->detail, sizeof(c->detail), "update_state: count=%d or null array", count);
        return ABYSS_ERR_INVALID_ARG;
    }
    for (int k = 0; k < count; ++k) {
        if (idx[k] < 0 || idx[k] >= c->state_n) {
            snprintf(c->detail, sizeof(c->detail), "update_state: index %d outside [0,%d)",
                     idx[k], c->state_n);
            return ABYSS_ERR_TARGET_RANGE;
        }
        for (int d = 0; d < 3; ++d)
            if (!std::isfinite(x[3 * k + d]) || !std::isfinite(v[3 * k + d]) || !std::isfinite(a[3 * k + d]) ||
                !std::isfinite(adot[3 * k + d])) {
                snprintf(c->detail, sizeof(c->detail), "update_state: non-finite data, k=%d", k);
                return ABYSS_ERR_INVALID_INPUT;
            }
        if (!std::isfinite(m[k]) || m[k] < 0.0 || !std::isfinite(t[k]) || std::isnan(r2[k]) || r2[k] < 0.0) {
            snprintf(c->detail, sizeof(c->detail), "update_state: bad m/t/r2, k=%d", k);
            return ABYSS_ERR_INVALID_INPUT;
        }
    }
    if (hipSetDevice(c->device) != hipSuccess) return ABYSS_ERR_HIP;
    // a captured update would read whatever the staging holds at its replays
    int rc = abyss::refuse_capture(c);
    if (rc != ABYSS_OK) return rc;
    // staging from a previous update may still be in flight
    if (c->busy_upd) {
        rc = abyss::ctx_wait(c);
        if (rc != ABYSS_OK) return rc;
    }
    const size_t rec_bytes = (size_t)count * kStateDoubles * sizeof(double);
    const size_t idx_bytes = ((size_t)count * sizeof(int) + 255) & ~size_t(255);
    const size_t need = rec_bytes + idx_bytes;
    if (need > c->upd_bytes) {
        if (c->h_upd) (void)hipHostFree(c->h_upd);
        c->h_upd = c->h_upd_dev = nullptr;
        c->upd_bytes = 0;
        const size_t cap = need + need / 2 + 4096;
        void *dev = nullptr;
        if (hipHostMalloc(&c->h_upd, cap, hipHostMallocMapped | hipHostMallocCoherent) !=
            hipSuccess)
            return ABYSS_ERR_OUT_OF_MEMORY;
        if (hipHostGetDevicePointer(&dev, c->h_upd, 0) != hipSuccess) return ABYSS_ERR_HIP;
        c->h_upd_dev = static_cast<char *>(dev);
        c->upd_bytes = cap;
    }
    int *hidx = reinterpret_cast<int *>(c->h_upd);
    double *hrec = reinterpret_cast<double *>(c->h_upd + idx_bytes);
    memcpy(hidx, idx, (size_t)count * sizeof(int));
    for (int k = 0; k < count; ++k) {
        double *r = hrec + (size_t)k * kStateDoubles;
        for (int d = 0; d < 3; ++d) {
            r[d] = x[3 * k + d];
            r[3 + d] = v[3 * k + d];
            r[6 + d] = a[3 * k + d];
            r[9 + d] = adot[3 * k + d];
        }
        r[12] = t[k];
        r[13] = m[k];
        r[14] = r2[k];
    }
    c->busy_upd = true;
    const char *src = c->h_upd_dev;
    hipLaunchKernelGGL(scatter_kernel, dim3((count + 63) / 64), dim3(256), 0, c->stream,
                       c->d_state, c->state_n, reinterpret_cast<const int *>(src),
                       reinterpret_cast<const double *>(src + idx_bytes), count);
    return hipGetLastError() == hipSuccess ? ABYSS_OK : ABYSS_ERR_HIP;
}

int abyss_ctx_predict(abyss_ctx_t c, double t_new)
{
    if (!c) return ABYSS_ERR_INVALID_ARG;
    if (c->state_n <= 0 || c->n != c->state_n) {
        snprintf(c->detail, sizeof(c->detail), "predict before upload_state");
        return ABYSS_ERR_NO_JSET;
    }
    if (!std::isfinite(t_new)) return ABYSS_ERR_INVALID_ARG;
    if (hipSetDevice(c->device) != hipSuccess) return ABYSS_ERR_HIP;
    const int n = c->state_n;
    double *jx = reinterpret_cast<double *>(c->d_j);
    float *m32 = reinterpret_cast<float *>(jx + 8 * (size_t)n);
    bool capturing = false;
    int rc = abyss::ctx_capturing(c, &capturing);
    if (rc != ABYSS_OK) return rc;
    // with resident lists in use, their gather records come from the same
    // pass (a pack of their own otherwise: 5 us at N = 65536); not when it is
    // being recorded, since nobody knows whether and when it will run
    if (capturing) c->predict_recorded = true;
    const bool records =
        !capturing && c->keep_lists && c->aos_bytes >= (size_t)n * sizeof(abyss::JRec);
    abyss::JRec *aos = records ? reinterpret_cast<abyss::JRec *>(c->d_aos) : nullptr;
    hipLaunchKernelGGL(predict_kernel, dim3((n + 255) / 256), dim3(256), 0, c->stream,
                       state_view(c->d_state, n), n, t_new, jx, m32, aos);
    c->jset_version += 1;
    if (hipGetLastError() != hipSuccess) return ABYSS_ERR_HIP;
    if (aos) c->aos_version = c->jset_version;
    return ABYSS_OK;
}

}  // extern "C"
