// Norm and populations by eigen-projection (src/hamiltonian.h:872-943, 1268-1307;
// src/process_output.cpp:332-355): for every distinct kappa the generalized
// eigenpairs H0(k) v = E S(k) v (S-orthonormal), and for every block r
// population_j = |v_j^H S(k_r) psi_r|^2, summed into the classes
// E < -c^2 (negative continuum), -c^2 <= E < 0 (bound) and E >= 0 (ionised).
// The eigenpairs are computed once per model on the host by this library's
// dense solver (gade_eig_dense: Cholesky, Householder tridiagonalization,
// implicit QL), one thread per distinct kappa, on the real parts of H0(k) and
// S(k) as the reference does (src/hamiltonian.h:906-943); the projections run
// in hand-written kernels.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <string>
#include <thread>
#include <vector>

#include "gade_device.h"
#include "gade_internal.h"

using gade::set_error;

namespace {

// per block r: w = S(k_r) psi_r (staged in LDS), then c_j = v_j . w for every eigenpair j of its kappa.
// COEF false: out[r][blockIdx.y] = (sums of |c_j|^2 over the classes for this workgroup's eigenpairs, psi_r^H S
// psi_r for the first); out may be pinned host memory.
// COEF true: out[r][j] = c_j, complex (the amplitudes behind the populations).
//
// One workgroup per block leaves most of the chip idle at the usual 60 to 500 blocks, and the work of one block
// is a chain of dependent memory reads, so latency bounds it: 256 threads with a thread per eigenpair and two
// loads in flight took 36.8 us at 104 blocks of 210 rows (57 us for the call).  Here 1024 threads take eight
// eigenpairs per wave, the sum over the rows split over eight lanes (64-byte row segments of V, the partial sums
// met by lane exchanges), and the first kBatch rows of each lane are read before w is formed, as they do not
// depend on it.  The rows of S are likewise split over eight lanes.  The eigenvectors are real and are stored so.
// Measured there: 17.6 us, and 30 us for the call with no copy and no allocation left in it (32 us with one
// workgroup per block, so that two passes follow each other).
constexpr int kLanes = 8;   // lanes that share one eigenpair's sum, or one row of S
constexpr int kBatch = 8;   // rows of V a lane holds in flight
constexpr int kEigThreads = 1024;
constexpr int kItems = kEigThreads / kLanes;
// workgroups per block: a pass of kItems eigenpairs each, while the blocks alone leave CUs without a workgroup
inline int eig_split(int nblk, int n) {
    return std::max(1, std::min((n + kItems - 1) / kItems, 512 / std::max(1, nblk)));
}
// threads of a workgroup: no more than the eigenpairs need, and 256 when there are more blocks than the chip holds
// workgroups of kEigThreads (two per CU): their phases then overlap instead of following each other.  Populations,
// us with kEigThreads throughout / now (one thread per eigenpair, the form before): 364 x 30: 26 / 19 (31); 1300 x 30:
// 49 / 25 (37-50); 1300 x 130: 77 / 64 (64); 544 x 130: 47 / 40 (52); 544 x 270: 83 / 80 (113).
inline int eig_threads(int nblk, int n) {
    return (std::min(n, nblk > 512 ? 32 : kItems) + 7) / 8 * 64;
}
template <bool COEF>
__global__ __launch_bounds__(kEigThreads) void k_eigproj(const double2 *__restrict__ x, const double2 *__restrict__ D,
                                                         const int *__restrict__ ell_col,
                                                         const int *__restrict__ blk_q, const double *__restrict__ VT,
                                                         const double *__restrict__ E, int n, int ellw, int nq,
                                                         double csq, double *__restrict__ out) {
    extern __shared__ double2 w[];
    __shared__ double sh[4 * (kEigThreads / 64)];
    const int r = blockIdx.x;
    const int q = blk_q[r];
    const int lane = threadIdx.x & 63, part = lane >> 3;
    const int item = (threadIdx.x >> 6) * 8 + (lane & 7);  // eigenpair (or row of S) of this lane's group
    const double *V = VT + (size_t)q * n * n;
    const int items = blockDim.x / kLanes;
    const int jf = blockIdx.y * items;  // first pass of this workgroup
    double v0[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; u++) {
        const int i = part + kLanes * u;
        v0[u] = (i < n && jf + item < n) ? V[(size_t)i * n + jf + item] : 0.0;
    }
    const double2 *Sq = D + ((size_t)2 * nq + q) * ellw * n;  // S(k) in ELL layout
    const double2 *xr = x + (size_t)r * n;
    double acc[4] = {0, 0, 0, 0};
    for (int a0 = 0; a0 < n; a0 += items) {
        const int a = a0 + item;
        double sx = 0, sy = 0;
        if (a < n) {
            double2 t = make_double2(0, 0);
            for (int sl = part; sl < ellw; sl += kLanes)
                t = cfma(Sq[(size_t)sl * n + a], xr[ell_col[(size_t)sl * n + a]], t);
            sx = t.x;
            sy = t.y;
        }
#pragma unroll
        for (int o = 8; o < 64; o <<= 1) {
            sx += __shfl_xor(sx, o, 64);
            sy += __shfl_xor(sy, o, 64);
        }
        if (a < n && part == 0) {
            w[a] = make_double2(sx, sy);
            if (!COEF && blockIdx.y == 0) {
                const double2 xa = xr[a];
                acc[3] += xa.x * sx + xa.y * sy;
            }
        }
    }
    __syncthreads();
    for (int j0 = jf; j0 < n; j0 += gridDim.y * items) {
        const int j = j0 + item;
        double cx = 0, cy = 0;
        if (j < n) {
            for (int i0 = 0; i0 < n; i0 += kLanes * kBatch) {
                if (i0 > 0 || j0 != jf) {
#pragma unroll
                    for (int u = 0; u < kBatch; u++) {
                        const int i = i0 + part + kLanes * u;
                        v0[u] = i < n ? V[(size_t)i * n + j] : 0.0;
                    }
                }
#pragma unroll
                for (int u = 0; u < kBatch; u++) {
                    const int i = i0 + part + kLanes * u;
                    if (i < n) {
                        const double2 wi = w[i];
                        cx = fma(v0[u], wi.x, cx);
                        cy = fma(v0[u], wi.y, cy);
                    }
                }
            }
        }
#pragma unroll
        for (int o = 8; o < 64; o <<= 1) {
            cx += __shfl_xor(cx, o, 64);
            cy += __shfl_xor(cy, o, 64);
        }
        if (j < n && part == 0) {
            if (COEF) {
                reinterpret_cast<double2 *>(out)[(size_t)r * n + j] = make_double2(cx, cy);
            } else {
                const double p = cx * cx + cy * cy;
                const double e = E[(size_t)q * n + j];
                if (e < -csq) acc[0] += p;
                else if (e < 0) acc[1] += p;
                else acc[2] += p;
            }
        }
    }
    if (!COEF) {
        block_sum<4>(acc, sh);
        if (threadIdx.x == 0)
            for (int k = 0; k < 4; k++) out[((size_t)r * gridDim.y + blockIdx.y) * 4 + k] = acc[k];
    }
}

}  // namespace

extern "C" {

int gade_eig_setup(gade_model_t *m) {
    if (!m) return GADE_EINVAL;
    if (m->d_evec) return GADE_OK;
    const int n = m->n, nq = m->nq, nnzb = m->nnzb;
    const size_t nn = (size_t)n * n;
    // radial values of s0..s2 and h00..h03 (real parts, as the reference's .real())
    std::vector<double2> hs((size_t)3 * nnzb), hh((size_t)4 * nnzb);
    GADE_HIP(hipMemcpy(hs.data(), m->d_s, sizeof(double2) * hs.size(), hipMemcpyDeviceToHost));
    GADE_HIP(hipMemcpy(hh.data(), m->d_h0, sizeof(double2) * hh.size(), hipMemcpyDeviceToHost));
    std::vector<double> E((size_t)nq * n), V((size_t)nq * nn);
    std::vector<int> rcs(nq, GADE_OK);
    std::atomic<int> next{0};
    auto worker = [&]() {
        std::vector<double> A(nn), B(nn);
        for (int q = next++; q < nq; q = next++) {
            const double k = m->kap_q[q];
            std::fill(A.begin(), A.end(), 0.0);
            std::fill(B.begin(), B.end(), 0.0);
            for (int i = 0; i < n; i++)
                for (int p = m->rad_Ap[i]; p < m->rad_Ap[i + 1]; p++) {
                    const int c = m->rad_Ai[p];
                    B[(size_t)i * n + c] = hs[p].x + k * hs[nnzb + p].x + k * k * hs[2 * nnzb + p].x;
                    A[(size_t)i * n + c] =
                        hh[p].x + k * hh[nnzb + p].x + k * k * hh[2 * nnzb + p].x + k * k * k * hh[3 * nnzb + p].x;
                }
            rcs[q] = gade_eig_dense(n, A.data(), B.data(), E.data() + (size_t)q * n, V.data() + (size_t)q * nn);
        }
    };
    const int nthr = std::max(1, std::min<int>(nq, std::min(16u, std::max(1u, std::thread::hardware_concurrency()))));
    std::vector<std::thread> pool;
    for (int t = 0; t < nthr; t++) pool.emplace_back(worker);
    for (auto &t : pool) t.join();
    for (int q = 0; q < nq; q++)
        if (rcs[q] != GADE_OK) {
            set_error("gade_eig_setup: generalized eigenproblem of kappa " + std::to_string(m->kap_q[q]) +
                      (rcs[q] == GADE_EINVAL ? " failed: S is not positive definite" : " did not converge"));
            return rcs[q];
        }
    // V[q][i][j] = v_j[i], as stored; h_eig receives the populations of every block
    double *d_eval = nullptr, *d_evec = nullptr, *h_eig = nullptr;
    GADE_TRY(gade::hip_alloc((void **)&d_eval, sizeof(double) * nq * n));
    int rc = gade::hip_alloc((void **)&d_evec, sizeof(double) * V.size());
    hipError_t e = hipSuccess;
    if (rc == GADE_OK) e = hipMemcpy(d_eval, E.data(), sizeof(double) * E.size(), hipMemcpyHostToDevice);
    if (rc == GADE_OK && e == hipSuccess) e = hipMemcpy(d_evec, V.data(), sizeof(double) * V.size(), hipMemcpyHostToDevice);
    if (rc == GADE_OK && e == hipSuccess)
        e = hipHostMalloc((void **)&h_eig, sizeof(double) * 4 * m->nblk * eig_split(m->nblk, n), hipHostMallocDefault);
    if (rc != GADE_OK || e != hipSuccess) {
        (void)hipFree(d_eval);
        if (d_evec) (void)hipFree(d_evec);
        if (rc != GADE_OK) return rc;
        set_error(std::string("gade_eig_setup: ") + hipGetErrorString(e));
        return GADE_EHIP;
    }
    m->h_eig = h_eig;
    m->d_eval = d_eval;
    m->d_evec = d_evec;
    return GADE_OK;
}

int gade_eig_values(gade_model_t *m, int *nkappa, int *kappa, double *energies) {
    if (!m) return GADE_EINVAL;
    GADE_TRY(gade_eig_setup(m));
    if (nkappa) *nkappa = m->nq;
    if (kappa) memcpy(kappa, m->kap_q.data(), sizeof(int) * m->nq);
    if (energies)
        GADE_HIP(hipMemcpy(energies, m->d_eval, sizeof(double) * m->nq * m->n, hipMemcpyDeviceToHost));
    return GADE_OK;
}

int gade_populations(gade_model_t *m, const double *x, double *norm, double *bound, double *ionised,
                     double *per_block) {
    if (!m || !x) return GADE_EINVAL;
    GADE_TRY(gade_eig_setup(m));
    const double csq = gade::kSoL * gade::kSoL;
    // the sums go straight to pinned host memory: four numbers per workgroup, read once the stream is done; calls of
    // several threads take turns, as they did on the stream
    std::lock_guard<std::mutex> one(m->eig_mutex);
    const int ny = eig_split(m->nblk, m->n);
    hipLaunchKernelGGL(k_eigproj<false>, dim3(m->nblk, ny), dim3(eig_threads(m->nblk, m->n)), sizeof(double2) * m->n, m->stream,
                       (const double2 *)x, m->d_D, m->d_ell_col, m->d_blk_q, m->d_evec, m->d_eval, m->n, m->ellw,
                       m->nq, csq, m->h_eig);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    if (e != hipSuccess) {
        set_error(std::string("gade_populations: ") + hipGetErrorString(e));
        return GADE_EHIP;
    }
    double tb = 0, ti = 0, tn = 0;
    for (int r = 0; r < m->nblk; r++) {
        double sum[4] = {0, 0, 0, 0};
        for (int y = 0; y < ny; y++)
            for (int k = 0; k < 4; k++) sum[k] += m->h_eig[((size_t)r * ny + y) * 4 + k];
        tb += sum[1];
        ti += sum[2];
        tn += sum[3];
        if (per_block) memcpy(per_block + (size_t)r * 4, sum, sizeof sum);
    }
    if (norm) *norm = tn;
    if (bound) *bound = tb;
    if (ionised) *ionised = ti;
    return GADE_OK;
}

int gade_psiev(gade_model_t *m, const double *x, double *psiev) {
    if (!m || !x || !psiev) return GADE_EINVAL;
    GADE_TRY(gade_eig_setup(m));
    const size_t cnt = (size_t)m->nblk * m->n;
    double2 *d_out = nullptr;
    GADE_TRY(gade::hip_alloc((void **)&d_out, sizeof(double2) * cnt));
    hipLaunchKernelGGL(k_eigproj<true>, dim3(m->nblk, eig_split(m->nblk, m->n)), dim3(eig_threads(m->nblk, m->n)),
                       sizeof(double2) * m->n, m->stream, (const double2 *)x, m->d_D, m->d_ell_col, m->d_blk_q, m->d_evec, m->d_eval, m->n, m->ellw,
                       m->nq, 0.0, (double *)d_out);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(psiev, d_out, sizeof(double2) * cnt, hipMemcpyDeviceToHost, m->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    (void)hipFree(d_out);
    if (e != hipSuccess) {
        set_error(std::string("gade_psiev: ") + hipGetErrorString(e));
        return GADE_EHIP;
    }
    // psiev_j = psi^H S v_j = conj(v_j^H S psi)  (src/hamiltonian.h:1318: psiseg.adjoint() * skev)
    for (size_t i = 0; i < cnt; i++) psiev[2 * i + 1] = -psiev[2 * i + 1];
    return GADE_OK;
}

// dense_write of src/dumpEigvals.cpp:87-108: int64 rows, int64 cols, then the column-major data
static int dense_write(const std::string &fname, int64_t rows, int64_t cols, const void *data, size_t elt) {
    FILE *fd = fopen(fname.c_str(), "wb");
    if (!fd) {
        set_error("cant open " + fname);
        return GADE_EIO;
    }
    bool ok = fwrite(&rows, sizeof rows, 1, fd) == 1 && fwrite(&cols, sizeof cols, 1, fd) == 1 &&
              fwrite(data, elt, (size_t)(rows * cols), fd) == (size_t)(rows * cols);
    ok = (fclose(fd) == 0) && ok;
    if (!ok) {
        set_error("write failed: " + fname);
        return GADE_EIO;
    }
    return GADE_OK;
}

int gade_eig_write(gade_model_t *m, const char *dir) {
    if (!m || !dir) return GADE_EINVAL;
    GADE_TRY(gade_eig_setup(m));
    const int n = m->n, nq = m->nq;
    const size_t nn = (size_t)n * n;
    std::vector<double> E((size_t)nq * n);
    std::vector<double> VT((size_t)nq * nn);
    std::vector<double2> evc(nn);
    GADE_HIP(hipMemcpy(E.data(), m->d_eval, sizeof(double) * E.size(), hipMemcpyDeviceToHost));
    GADE_HIP(hipMemcpy(VT.data(), m->d_evec, sizeof(double) * VT.size(), hipMemcpyDeviceToHost));
    for (int q = 0; q < nq; q++) {
        const int kappa = m->kap_q[q];
        GADE_TRY(dense_write(std::string(dir) + "/evl" + std::to_string(kappa) + ".mat", n, 1, E.data() + (size_t)q * n,
                             sizeof(double)));
        // column j = eigenvector j: evc[j * n + i] = v_j[i] (the files hold complex numbers)
        const double *V = VT.data() + (size_t)q * nn;
        for (int i = 0; i < n; i++)
            for (int j = 0; j < n; j++) evc[(size_t)j * n + i] = make_double2(V[(size_t)i * n + j], -0.0);
        GADE_TRY(dense_write(std::string(dir) + "/evc" + std::to_string(kappa) + ".mat", n, n, evc.data(),
                             sizeof(double2)));
    }
    return GADE_OK;
}

}  // extern "C"
