// Start-up derivatives and neighbour-radius adaptation on the device
// (include/abyss_regf.h: abyss_ctx_derivs23, abyss_ctx_update_radius).
//
// ABYSS computes the second and third time derivatives of every particle's
// acceleration once at start-up, by an O(N^2) host loop per particle split
// into regular and irregular parts (CalculateAcceleration23,
// src_mpi/Particle/Initialize.cpp:102-185), and rescales each particle's
// neighbour radius after every regular step from its neighbour count
// (Particle::updateRadius, src_mpi/Particle/UpdateParticle.cpp:108-139).
// Both run here on the resident particle state (abyss_ctx_upload_state).
//
// derivs23: one target per lane; every lane of a wave walks the same j, so
// the j record (x, v, a, adot, m; 128-byte AoS copy of the state) is read at
// a wave-uniform address and reaches the lanes through the scalar cache.
// The four waves of a workgroup share 64 targets and take a quarter of the
// workgroup's j range each; the j range is split over grid.y as well, so
// that small target blocks still fill the chip.  Partial sums are added in a
// fixed order (bitwise reproducible).
#include "regf_context.h"

#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <cmath>

namespace {

struct __align__(128) DRec {
    double x, y, z, vx, vy, vz, ax, ay, az, jx, jy, jz, m, pad0, pad1, pad2;
};

// State SoA (stride n): x[3][n], v[3][n], a[3][n], ad[3][n], t[n], m[n], r2[n].
__global__ __launch_bounds__(256) void pack_drec_kernel(const double *__restrict__ st, int n,
                                                        DRec *__restrict__ out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t N = (size_t)n;
    out[i] = DRec{st[i],          st[N + i],      st[2 * N + i],  st[3 * N + i],
                  st[4 * N + i],  st[5 * N + i],  st[6 * N + i],  st[7 * N + i],
                  st[8 * N + i],  st[9 * N + i],  st[10 * N + i], st[11 * N + i],
                  st[13 * N + i], 0.0,            0.0,            0.0};
}

// One split of the j range for 64 targets.  The terms are the reference's
// (x, v, da = a_j - a_i, dj = adot_j - adot_i, w = m/r^3, q = 1/r^2, p = -1
// for REF, whose projections x.(a_i - a_j)/r2, v.(a_i - a_j)/r2 and
// x.(adot_i - adot_j)/r2 enter B and C, p = 1 for the exact derivatives of
// m x/|x|^3 along the relative orbit), collected by vector:
//   A = (x.v) q,  T = (v.v + p x.da) q,  D = p (3 v.da + x.dj) q
//   a2 = w da - 6 w A v + w (15 A^2 - 3 T) x
//   a3 = w dj - 9 w A da + 3 w (15 A^2 - 3 T) v + w (A (45 T - 105 A^2) - 3 D) x
// which is the reference's B = T + A^2, C = D + A (3 B - 4 A^2) inserted into
// adot2 = w da - 6 A f1 - 3 B f0, adot3 = w dj - 9 A adot2 - 9 B f1 - 3 C f0.
// Bound by FP64 VALU issue: 81 instructions per pair with one hardware
// reciprocal root (refined to second order) and no division; the j records
// cost no vector instruction.  Written term by term (8 divisions and a square
// root per pair, one wave walking at least 1024 j) a call took 2194 us at
// N = m = 16384 and 1022 us at N = 40000, m = 1; now 841 and 47 us.
// A step with a neighbour, the target itself or an r^2 whose r^-3 is zero
// takes a branch that moves those lanes' terms to the irregular sums (or
// drops them) and zeroes their factors.
template <bool REF>
__global__ __launch_bounds__(256) void derivs23_kernel(const DRec *__restrict__ jr, int n,
                                                       const int *__restrict__ tgt, int nt,
                                                       const double *__restrict__ rnb2,
                                                       int jspan, double *__restrict__ part)
{
    __shared__ double s_sum[3][12][64];   // waves 1 to 3 hand their sums to wave 0
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = blockIdx.x * 64 + lane;
    const int s = blockIdx.y;
    // this wave's quarter of the split (empty for the last waves of a short one)
    const int sub = (jspan + 3) / 4;
    const int j0 = s * jspan + wave * sub;
    const int j1 = min(min(n, (s + 1) * jspan), j0 + sub);
    const bool active = q < nt;
    const int i = active ? tgt[q] : 0;
    const DRec ri = jr[i];
    const double rn = active ? rnb2[i] : -1.0;
    double reg[6] = {0, 0, 0, 0, 0, 0}, irr[6] = {0, 0, 0, 0, 0, 0};   // a2, a3
    // r^-3 of anything above is below the smallest double
    constexpr double kFar = 1.0e290;
    auto pair = [&](const DRec &rj) {
        const double x[3] = {rj.x - ri.x, rj.y - ri.y, rj.z - ri.z};
        const double v[3] = {rj.vx - ri.vx, rj.vy - ri.vy, rj.vz - ri.vz};
        const double da[3] = {rj.ax - ri.ax, rj.ay - ri.ay, rj.az - ri.az};
        const double dj[3] = {rj.jx - ri.jx, rj.jy - ri.jy, rj.jz - ri.jz};
        auto dot = [](const double *a, const double *b) {
            return fma(a[2], b[2], fma(a[1], b[1], a[0] * b[0]));
        };
        const double r2 = dot(x, x);
        const double xa = dot(x, da), xj = dot(x, dj), va = dot(v, da);
        double y = __builtin_amdgcn_rsq(r2);
        const double e = fma(-(r2 * y), y, 1.0);
        y = fma(y * fma(0.375, e, 0.5), e, y);
        const double iq = y * y;
        double w = rj.m * y * iq;
        const double A = dot(v, x) * iq;
        const double T = (REF ? dot(v, v) - xa : dot(v, v) + xa) * iq;
        const double D = (REF ? -fma(3.0, va, xj) : fma(3.0, va, xj)) * iq;
        const double A2 = A * A;
        const double wA = w * A;
        double cv = -6.0 * wA, cd = -9.0 * wA;
        double cx = w * fma(15.0, A2, -3.0 * T);
        double cy = w * fma(A, fma(45.0, T, -105.0 * A2), -3.0 * D);
        const bool near = !(r2 > rn);
        auto add = [&](double *o) {
            const double cw = 3.0 * cx;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                o[d] = fma(cx, x[d], fma(cv, v[d], fma(w, da[d], o[d])));
                o[3 + d] = fma(cy, x[d], fma(cw, v[d], fma(cd, da[d], fma(w, dj[d], o[3 + d]))));
            }
        };
        if (__any(near || !(r2 < kFar))) {
            const bool none = r2 == 0.0 || !(r2 < kFar);   // self, coincident, out of reach
            if (none) w = cv = cd = cx = cy = 0.0;
            if (near) {
                add(irr);
                w = cv = cd = cx = cy = 0.0;
            }
        }
        add(reg);
    };
    if (j0 < j1) {
        DRec rj = jr[j0];   // wave-uniform address
        for (int j = j0; j < j1; ++j) {
            const DRec next = jr[min(j + 1, j1 - 1)];
            pair(rj);
            rj = next;
        }
    }
    if (wave > 0)
#pragma unroll
        for (int c = 0; c < 12; ++c) s_sum[wave - 1][c][lane] = c < 6 ? reg[c] : irr[c - 6];
    __syncthreads();
    if (wave > 0 || !active) return;
    double *o = part + ((size_t)s * nt + q) * 12;
#pragma unroll
    for (int c = 0; c < 12; ++c) {
        double a = c < 6 ? reg[c] : irr[c - 6];
        for (int k = 0; k < 3; ++k) a += s_sum[k][c][lane];
        o[c] = a;
    }
}

// out[e] = sum over the splits of part[s][e]: 16 threads per element take the
// splits s, s + 16, ... in order, and their sums are added in order.
__global__ __launch_bounds__(256) void derivs_sum_kernel(const double *__restrict__ part, int S,
                                                         int nt, double *__restrict__ out)
{
    __shared__ double s_sum[16][16];
    const int k = threadIdx.x >> 4, c = threadIdx.x & 15;
    const size_t e = (size_t)blockIdx.x * 16 + c;
    const size_t total = (size_t)nt * 12;
    double acc = 0.0;
    if (e < total)
        for (int s = k; s < S; s += 16) acc += part[(size_t)s * total + e];
    s_sum[k][c] = acc;
    __syncthreads();
    if (k > 0 || e >= total) return;
    for (int t = 1; t < 16; ++t) acc += s_sum[t][c];
    out[e] = acc;
}

// Radius rule of the reference on r2 (the squared radius) for the targets
// of the last launch, from their neighbour counts (|count| if overflowed);
// contraction off, so it equals the host rule bit for bit.
#pragma clang fp contract(off)
__global__ __launch_bounds__(256) void update_radius_kernel(const int *__restrict__ tgt, int nt,
                                                            const int *__restrict__ nnb, int fix,
                                                            int nmax, double *__restrict__ st_r2,
                                                            double *__restrict__ j_r2,
                                                            double *__restrict__ r2_out)
{
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nt) return;
    const int i = tgt[q];
    const int c = nnb[q] < 0 ? -nnb[q] : nnb[q];
    double r2 = j_r2[i];
    const double cc = (double)(nmax - fix);
    const double x = (double)(c - fix);
    if (c > fix) r2 *= (1. - 0.9 / (cc * cc) * fabs(x) * x);
    else if (c < fix) r2 *= (1. - 0.5 / (cc * cc * cc) * (x * x * x));
    j_r2[i] = r2;
    if (st_r2) st_r2[i] = r2;
    r2_out[q] = r2;
}
#pragma clang fp contract(on)

int ensure_buf(char **d, size_t *bytes, size_t need, hipStream_t st)
{
    if (need <= *bytes) return ABYSS_OK;
    if (hipStreamSynchronize(st) != hipSuccess) return ABYSS_ERR_HIP;
    if (*d) (void)hipFree(*d);
    *d = nullptr;
    *bytes = 0;
    if (hipMalloc(d, need) != hipSuccess) return ABYSS_ERR_OUT_OF_MEMORY;
    *bytes = need;
    return ABYSS_OK;
}

}  // namespace

extern "C" {

int abyss_ctx_derivs23(abyss_ctx_t c, int nt, const int *targets, int reference_signs,
                       double *out)
{
    if (!c) return ABYSS_ERR_INVALID_ARG;
    if (c->state_n <= 0 || c->n != c->state_n) {
        snprintf(c->detail, sizeof(c->detail), "derivs23 needs abyss_ctx_upload_state first");
        return ABYSS_ERR_NO_JSET;
    }
    if (nt <= 0 || !targets || !out) {
        snprintf(c->detail, sizeof(c->detail), "derivs23: nt=%d or null array", nt);
        return ABYSS_ERR_INVALID_ARG;
    }
    const int n = c->state_n;
    for (int k = 0; k < nt; ++k)
        if (targets[k] < 0 || targets[k] >= n) {
            snprintf(c->detail, sizeof(c->detail), "derivs23: target %d outside [0,%d)",
                     targets[k], n);
            return ABYSS_ERR_TARGET_RANGE;
        }
    if (hipSetDevice(c->device) != hipSuccess) return ABYSS_ERR_HIP;
    // j splits: 16 workgroups per CU, each split at least 64 j (16 per wave)
    const int gx = (nt + 63) / 64;
    const int cu = c->cu_count > 0 ? c->cu_count : 256;
    int S = std::max(1, (cu * 16 + gx - 1) / gx);
    S = std::min(S, std::max(1, n / 64));
    S = std::min(S, 1024);
    const int jspan = (n + S - 1) / S;
    S = (n + jspan - 1) / jspan;
    const size_t rec_bytes = (size_t)n * sizeof(DRec);
    const size_t part_bytes = (size_t)S * nt * 12 * sizeof(double);
    const size_t tgt_bytes = (((size_t)nt * sizeof(int)) + 255) & ~size_t(255);
    const size_t out_bytes = (size_t)nt * 12 * sizeof(double);
    int rc = ensure_buf(&c->d_drv, &c->drv_bytes, rec_bytes + part_bytes + tgt_bytes, c->stream);
    if (rc != ABYSS_OK) return rc;
    if (hipStreamSynchronize(c->stream) != hipSuccess) return ABYSS_ERR_HIP;
    if (out_bytes + tgt_bytes > c->h_drv_bytes) {
        if (c->h_drv) (void)hipHostFree(c->h_drv);
        c->h_drv = nullptr;
        c->h_drv_bytes = 0;
        if (hipHostMalloc(&c->h_drv, out_bytes + tgt_bytes,
                          hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess)
            return ABYSS_ERR_OUT_OF_MEMORY;
        c->h_drv_bytes = out_bytes + tgt_bytes;
    }
    void *h_dev = nullptr;
    if (hipHostGetDevicePointer(&h_dev, c->h_drv, 0) != hipSuccess) return ABYSS_ERR_HIP;
    // the sums go straight into the mapped block, so no copy follows them
    double *d_out = reinterpret_cast<double *>(static_cast<char *>(h_dev) + tgt_bytes);
    DRec *d_rec = reinterpret_cast<DRec *>(c->d_drv);
    double *d_part = reinterpret_cast<double *>(c->d_drv + rec_bytes);
    int *d_tgt = reinterpret_cast<int *>(c->d_drv + rec_bytes + part_bytes);
    memcpy(c->h_drv, targets, (size_t)nt * sizeof(int));
    if (hipMemcpyAsync(d_tgt, c->h_drv, (size_t)nt * sizeof(int), hipMemcpyHostToDevice,
                       c->stream) != hipSuccess)
        return ABYSS_ERR_HIP;
    hipLaunchKernelGGL(pack_drec_kernel, dim3((n + 255) / 256), dim3(256), 0, c->stream,
                       c->d_state, n, d_rec);
    const double *st_r2 = c->d_state + 14 * (size_t)n;
    if (reference_signs)
        hipLaunchKernelGGL(derivs23_kernel<true>, dim3(gx, S), dim3(256), 0, c->stream, d_rec, n,
                           d_tgt, nt, st_r2, jspan, d_part);
    else
        hipLaunchKernelGGL(derivs23_kernel<false>, dim3(gx, S), dim3(256), 0, c->stream, d_rec,
                           n, d_tgt, nt, st_r2, jspan, d_part);
    const size_t total = (size_t)nt * 12;
    hipLaunchKernelGGL(derivs_sum_kernel, dim3((unsigned)((total + 15) / 16)), dim3(256), 0,
                       c->stream, d_part, S, nt, d_out);
    if (hipGetLastError() != hipSuccess) return ABYSS_ERR_HIP;
    double *h_out = reinterpret_cast<double *>(c->h_drv + tgt_bytes);
    if (hipStreamSynchronize(c->stream) != hipSuccess) return ABYSS_ERR_HIP;
    memcpy(out, h_out, out_bytes);
    return ABYSS_OK;
}

int abyss_ctx_update_radius(abyss_ctx_t c, int fix, int nmax, double *r2_out)
{
    if (!c) return ABYSS_ERR_INVALID_ARG;
    if (c->n <= 0 || c->nt <= 0 || !c->counts_valid) {
        snprintf(c->detail, sizeof(c->detail), "update_radius: no launch to take counts from");
        return ABYSS_ERR_NO_JSET;
    }
    if (fix < 0 || nmax <= fix || !r2_out) {
        snprintf(c->detail, sizeof(c->detail), "update_radius: fix=%d nmax=%d or null output",
                 fix, nmax);
        return ABYSS_ERR_INVALID_ARG;
    }
    if (hipSetDevice(c->device) != hipSuccess) return ABYSS_ERR_HIP;
    const int nt = c->nt;
    int rc = ensure_buf(&c->d_rad, &c->rad_bytes, (size_t)nt * sizeof(double), c->stream);
    if (rc != ABYSS_OK) return rc;
    double *j_r2 = reinterpret_cast<double *>(c->d_j) + 7 * (size_t)c->n;   // j-set r_nb^2
    double *st_r2 = (c->state_n == c->n && c->d_state) ? c->d_state + 14 * (size_t)c->n : nullptr;
    double *d_r2 = reinterpret_cast<double *>(c->d_rad);
    hipLaunchKernelGGL(update_radius_kernel, dim3((nt + 255) / 256), dim3(256), 0, c->stream,
                       c->tgt, nt, c->d_nnb, fix, nmax, st_r2, j_r2, d_r2);
    if (hipGetLastError() != hipSuccess) return ABYSS_ERR_HIP;
    if (hipMemcpyAsync(r2_out, d_r2, (size_t)nt * sizeof(double), hipMemcpyDeviceToHost,
                       c->stream) != hipSuccess ||
        hipStreamSynchronize(c->stream) != hipSuccess)
        return ABYSS_ERR_HIP;
    return ABYSS_OK;
}

}  // extern "C"
