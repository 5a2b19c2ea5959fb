// Batched small DOCI solves, every request of a batch in lock step (see batch.hip).
#pragma once

#include "common.h"

namespace cf {

constexpr int kBatchMaxL = 32;        // orbitals
constexpr int kBatchMaxSteps = 400;   // Lanczos steps (products) per request
constexpr int kBatchRunning = 1 << 30;  // no step has given a result yet

// One request of a batch (device memory).
struct DociBatchJob {
    const double* h = nullptr;     // L x L (rotated) one-electron integrals
    const double* V = nullptr;     // L^4 physics two-electron integrals
    const str_t* s = nullptr;      // the n pair strings of the (L, np) space, rank order
    const uint32_t* hops = nullptr; // packed hops [np * nv][n] of that space (launch_doci_hops)
    double tol = 1e-12;            // ||r|| <= tol |theta|
    double tol_energy = 0.0;       // Kato-Temple estimate stop (0: off)
    uint64_t seed = 0;             // start vector
    double* out = nullptr;         // eigval, residual, products, status (0 converged, 1 step limit)
    double* scratch = nullptr;     // doci_batch_scratch(n, L) doubles
    int* done = nullptr;           // step whose launch gave the request its result (before: kBatchRunning)
    int L = 0, np = 0, nv = 0, n = 0;
    int check = 2;                 // convergence test every `check` steps (>= 1)
    int max_steps = kBatchMaxSteps;
};

// Largest DOCI space a batch takes.
int doci_batch_capacity();
// Doubles of scratch of one request: diagonal, two images H v, three Krylov
// vectors, the coefficients alpha and beta, the hop elements.
inline uint64_t doci_batch_scratch(uint64_t n, int L) {
    return 6 * n + 2 * (uint64_t)(kBatchMaxSteps + 2) + (uint64_t)L * L;
}
// Hop columns (launch_doci_ell_fill, [np * nv][n]) packed in place with the
// element each takes: (j L + k) << 20 | rank << 3.
void launch_doci_hops(const str_t* s, uint64_t n, int L, int np, uint32_t* col, hipStream_t st);
// Solves `count` requests of at most max_n determinants and max_L orbitals
// (max_n picks the workgroup shape).  `left` is a device counter and `flag` a
// page-locked host word that the device can write; returns once every
// request has its result (ordered on s).
void run_doci_batch(const DociBatchJob* d_jobs, int count, int max_n, int max_L, int max_steps, int* left,
                    volatile int* flag, hipEvent_t ev[2], hipStream_t s);

}  // namespace cf
