// Many small DOCI ground-state solves at once: the served stream's small
// requests (DOCI spaces of up to 13,312 determinants, L <= 16 at half
// filling), which the reference solves one after another
// (OrbitalOptimization::update_cim -> set_ham -> build_ci -> solve,
// SimulatedAnnealing.cpp:83-87, CIMethod.cpp:117-126,241-268).
//
// The DOCI matrix of DOCI::construct_CI_matrix (CIMethod.cpp:611-660) is
// applied without storing it -- the diagonal 2 sum h_ii + sum_i (ii|ii) +
// sum_{k != l} (2 (kk|ll) - (kl|lk)) per row once, and the pair hops j -> k with
// element V(j,j,k,k) -- in plain FP64 Lanczos, and every request of the batch
// takes its step j in one launch:
//   * a request's rows are split over `nchunk` workgroups.  Each of them reads
//     the whole of H v_{j-1}, v_{j-1} and v_{j-2} (a few times n doubles from
//     L2), forms alpha_{j-1}, the next vector and its norm itself, so that no
//     workgroup waits for another, holds v_j in LDS and applies H to its own
//     rows.  The sums run over a fixed thread mapping of all n rows, so a
//     request's result depends neither on the split nor on the batch.
//   * one more workgroup per request tests T_{j-1} for convergence meanwhile:
//     one wave finds the lowest eigenvalue and another the second by
//     Sturm-count multisection, each then the last component of its
//     eigenvector, and the solver's stopping tests are ||r_0|| = |beta_m z_m|
//     <= tol |theta_0|, or the Kato-Temple estimate ||r_0||^2 / (theta_1 -
//     ||r_1|| - theta_0) <= tol_energy.  Without reorthogonalisation converged
//     Ritz values reappear as copies; a second value within 1e-10 |theta_0| of
//     the first is such a copy and the gap is taken to the next distinct one.
// The host stays eight steps ahead and stops when the last request is done.
//
// What bounds it: a step is the latency of one launch, two reductions over n
// and np nv dependent-free gathers a row.  One workgroup per request, with the
// test on one of its waves, left most CUs idle and waited for a column from L2
// at every hop: 48 requests of L=14 (3,432 rows) took 9.1 ms on 48 of 256 CUs;
// now a step is 14.5 us on average, its test beside it, and the batch 1.4 ms (a
// whole call 10.9 -> 2.7 ms, the rest of it the integrals' way to the GPU).
#include "batch.h"

#include <algorithm>

namespace cf {

namespace {

constexpr int kMaxSteps = kBatchMaxSteps;

__device__ __forceinline__ double wave_sum64(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// T_m of one convergence test, scaled to [-1, 1] by its Gershgorin bounds and
// padded to whole blocks of kBlk elements, which are read from LDS together.
// Signs are compared as sign bits: as conditions they went through the scalar
// unit, and an element of a test cost 0.65 us instead of 0.1.
constexpr int kBlk = 16;
constexpr int kPadSteps = (kMaxSteps + kBlk - 1) / kBlk * kBlk;
struct alignas(16) TestMatrix {
    double a[kPadSteps];   // diagonal (padding 4: no sign change)
    double b2[kPadSteps];  // b_{i-1}^2, the square of the element before
    // from the last row to the first (element q is row i = m - 1 - q)
    double ra[kPadSteps];  // diagonal
    double rn[kPadSteps];  // b_i
    double rb[kPadSteps];  // 1 / b_{i-1} (0 at row 0 and in the padding)
};

// Eigenvalues of T_m below x: sign changes of the leading minors p_0 .. p_m,
// p_i = (a_i - x) p_{i-1} - b_{i-1}^2 p_{i-2} (one dependent FMA an element; a
// zero counts as positive, its successor has the sign opposite to its
// predecessor's, so the changes add up).
__device__ __forceinline__ int sturm_count(const TestMatrix& T, int m, double x) {
    int c = 0, sign = 0;
    double pp = 0.0, p = 1.0;
    for (int i0 = 0; i0 < m; i0 += kBlk) {
        double a[kBlk], b2[kBlk];
#pragma unroll
        for (int q = 0; q < kBlk; ++q) {
            a[q] = T.a[i0 + q] - x;
            b2[q] = T.b2[i0 + q];
        }
#pragma unroll
        for (int q = 0; q < kBlk; ++q) {
            const double pn = fma(a[q], p, -(b2[q] * pp));
            pp = p;
            p = pn;
            const int sg = __double2hiint(pn);
            c += (int)((unsigned)(sg ^ sign) >> 31);
            sign = sg;
        }
        const double big = fmax(fabs(p), fabs(pp));  // a block multiplies by 5^16 at most
        const double sc = big > 1e100 ? 1e-100 : big < 1e-100 ? 1e100 : 1.0;
        p *= sc;
        pp *= sc;
    }
    return c;
}

// k-th smallest eigenvalue (k = 0, 1, ...) of T_m by multisection over one
// wave: every lane tests one point, the bracket shrinks 65-fold per round.
// `prev`: that eigenvalue of an earlier T (any value above 1: none).  It is an
// upper bound (interlacing), and the first round's points lie at distances
// below it that grow 1.75-fold from lane to lane, so near convergence four
// rounds are saved.  The value is taken to rounding (two units of the last
// place): the last component moves by a hundred times its error, 5e-12 of the
// residual estimate when it was taken to 1e-13, 3e-14 now, as much as the
// rounding of T moves it.
__device__ double kth_eigenvalue(const TestMatrix& T, int m, int k, double prev) {
    const int lane = threadIdx.x & 63;
    double lo = -1.0, hi = 1.0;
    const bool warm = prev < 1.0;
    for (int round = 0; round < 13 && hi - lo > 2.5e-16; ++round) {
        const bool w = warm && round == 0;
        const double x = w ? prev - exp2(1.0 - 51.0 * (double)lane / 63.0) : lo + (hi - lo) * (double)(lane + 1) / 65.0;
        // the first lane whose point has more than k eigenvalues below it
        const unsigned long long ball = __ballot(sturm_count(T, m, x) > k);
        const int first = ball ? __builtin_ctzll(ball) : 64;
        const double nlo = first > 0 ? __shfl(x, first - 1, 64) : lo;
        const double nhi = first < 64 ? __shfl(x, first < 64 ? first : 63, 64) : w ? fmin(1.0, prev + 2e-13) : hi;
        lo = fmax(lo, nlo);
        hi = nhi;
    }
    return 0.5 * (lo + hi);
}

// |last component| of the normalised eigenvector of T_m for eigenvalue x by
// the recurrence from its end, z_{i-1} = -((a_i - x) z_i + b_i z_{i+1}) /
// b_{i-1}: the component is small and the others grow from it, which is the
// stable direction; only a few digits are needed.
__device__ __forceinline__ double last_component(const TestMatrix& T, int m, double x) {
    double zn = 0.0, z = 1.0, last = 1.0, nrm = 1.0;
    for (int i0 = 0; i0 < m; i0 += kBlk) {
        double a[kBlk], b[kBlk], rb[kBlk];
#pragma unroll
        for (int q = 0; q < kBlk; ++q) {
            a[q] = T.ra[i0 + q] - x;
            b[q] = T.rn[i0 + q];
            rb[q] = T.rb[i0 + q];
        }
#pragma unroll
        for (int q = 0; q < kBlk; ++q) {
            const double zp = -fma(a[q], z, b[q] * zn) * rb[q];
            zn = z;
            z = zp;
            nrm = fma(z, z, nrm);
            if (q % 4 == 3) {  // an element grows by 2e14 at most (beta > 1e-14 |alpha|)
                const double sc = nrm > 1e100 ? 1e-50 : 1.0;
                z *= sc;
                zn *= sc;
                last *= sc;
                nrm *= sc * sc;
            }
        }
    }
    return nrm < 1e300 ? last / sqrt(nrm) : 0.0;  // not finite: no residual
}

__device__ __forceinline__ double start_value(uint64_t seed, uint64_t q) {
    uint64_t z = seed + 0x9E3779B97F4A7C15ULL * (q + 1);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    z ^= z >> 31;
    return 1.0 + 0.5 * ((double)(z >> 11) * (1.0 / 9007199254740992.0) - 0.5);
}

}  // namespace

namespace {

// Block sum over NT threads in a fixed order.
template <int NT>
__device__ __forceinline__ double block_sum(double v, double* red) {
    v = wave_sum64(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) s += red[i];
    __syncthreads();
    return s;
}

// The parts of a request's scratch.
struct Work {
    double *dg, *u, *v, *al, *be, *hop;
    __device__ explicit Work(const DociBatchJob& J) {
        const size_t n = (size_t)J.n;
        dg = J.scratch;
        u = dg + n;
        v = u + 2 * n;
        al = v + 3 * n;
        be = al + kMaxSteps + 2;
        hop = be + kMaxSteps + 2;
    }
};

// Convergence test of T_m, m = j - 1, by the whole workgroup (two waves work);
// sets the request's result and the step it was found in when it stops.
__device__ void lanczos_test(const DociBatchJob& J, int j, int maxs, TestMatrix& T, int count, int* left, int* flag) {
    const int m = j - 1;
    const Work W(J);
    __shared__ double ctl[6];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const double alpha = W.al[m - 1], beta = W.be[m - 1];
    const bool broke = !(beta > 1e-14 * fabs(alpha));
    if (!((m >= 4 && m % J.check == 0) || m == maxs || broke)) return;
    double glo = 1e300, ghi = -1e300;  // Gershgorin bounds, in every wave
    for (int i = lane; i < m; i += 64) {
        const double rad = (i > 0 ? fabs(W.be[i - 1]) : 0.0) + (i < m - 1 ? fabs(W.be[i]) : 0.0);
        glo = fmin(glo, W.al[i] - rad);
        ghi = fmax(ghi, W.al[i] + rad);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        glo = fmin(glo, __shfl_xor(glo, off, 64));
        ghi = fmax(ghi, __shfl_xor(ghi, off, 64));
    }
    const double pad = 1e-12 * fmax(1.0, fmax(fabs(glo), fabs(ghi)));
    const double mid = 0.5 * (glo + ghi), half = 0.5 * (ghi - glo) + pad, rh = 1.0 / half;
    for (int i = tid; i < (m + kBlk - 1) / kBlk * kBlk; i += blockDim.x) {
        const double bl = i > 0 && i < m ? W.be[i - 1] * rh : 0.0;
        T.a[i] = i < m ? (W.al[i] - mid) * rh : 4.0;
        T.b2[i] = bl * bl;
        const int q = m - 1 - i;  // row of element i counted from the end
        const double bp = q > 0 ? W.be[q - 1] * rh : 0.0;
        T.ra[i] = q >= 0 ? (W.al[q] - mid) * rh : 0.0;
        T.rn[i] = i > 0 && q >= 0 ? W.be[q] * rh : 0.0;
        T.rb[i] = bp != 0.0 ? 1.0 / bp : 0.0;
    }
    __syncthreads();
    double* last_th = W.al + kMaxSteps;  // theta_0 and theta_1 of the last test
    if (wv < 2 && wv < m) {  // theta_0 and theta_1 at the same time
        const double xk = kth_eigenvalue(T, m, wv, (last_th[wv] - mid) * rh);
        if (lane == 0) {
            ctl[wv] = xk;
            last_th[wv] = mid + half * xk;
        }
    }
    __syncthreads();
    const double x0 = ctl[0], th0 = mid + half * x0;
    double x1 = m > 1 ? ctl[1] : x0;
    bool have1 = m > 1;
    int k1 = 1;
    while (have1 && half * (x1 - x0) <= 1e-10 * fmax(1.0, fabs(th0))) {  // copies of theta_0 skipped
        __syncthreads();
        if (++k1 >= m || k1 >= 6) {
            have1 = false;
            break;
        }
        if (wv == 0) {
            const double xk = kth_eigenvalue(T, m, k1, 2.0);
            if (lane == 0) ctl[1] = xk;
        }
        __syncthreads();
        x1 = ctl[1];
    }
    if (lane == 0 && wv < 2) ctl[2 + wv] = beta * last_component(T, m, wv == 0 ? x0 : x1);
    __syncthreads();
    const double r0 = ctl[2], r1 = ctl[3], th1 = mid + half * x1;
    bool stop = r0 <= J.tol * fabs(th0) || broke;
    if (!stop && J.tol_energy > 0.0 && have1) {
        const double mu = th1 - r1;
        stop = mu > th0 && r0 * r0 <= J.tol_energy * (mu - th0);
    }
    if ((stop || m == maxs) && tid == 0) {
        J.out[0] = th0;
        J.out[1] = r0;
        J.out[2] = (double)m;
        J.out[3] = stop ? 0.0 : 1.0;
        __hip_atomic_store(J.done, j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (atomicAdd(left, 1) + 1 == count) {
            *flag = 1;  // host memory
            __threadfence_system();
        }
    }
}

}  // namespace

__global__ void __launch_bounds__(256) k_doci_hops(const str_t* __restrict__ s, uint64_t n, int L, int np,
                                                   uint32_t* __restrict__ col) {
    const uint64_t r = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (r >= n) return;
    const str_t full = L >= 64 ? ~(str_t)0 : ((str_t)1 << L) - 1;
    str_t o = s[r];
    const str_t vir = ~o & full;
    uint64_t t = 0;
    for (int a = 0; a < np; ++a) {
        const int j = 63 - __builtin_clzll(o);
        o ^= (str_t)1 << j;
        for (str_t v = vir; v;) {
            const int k = 63 - __builtin_clzll(v);
            v ^= (str_t)1 << k;
            uint32_t* e = col + t * n + r;
            *e = (uint32_t)(j * L + k) << 20 | *e << 3;
            ++t;
        }
    }
}

void launch_doci_hops(const str_t* s, uint64_t n, int L, int np, uint32_t* col, hipStream_t st) {
    if (!n) return;
    CF_REQUIRE(L <= kBatchMaxL && n <= (uint64_t)doci_batch_capacity(), "packed hops: L <= 32, n <= 13312");
    k_doci_hops<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(s, n, L, np, col);
    CF_HIP(hipGetLastError());
}

// Diagonal and hop elements of every request; the request is not done.
__global__ void __launch_bounds__(256) k_doci_batch_init(const DociBatchJob* __restrict__ jobs, int* left) {
    __shared__ double pd[kBatchMaxL * kBatchMaxL];  // 2 (kk|ll) - (kl|lk), k != l
    __shared__ double d1[kBatchMaxL];               // 2 h_ii + (ii|ii)
    const DociBatchJob J = jobs[blockIdx.y];
    const Work W(J);
    const int L = J.L;
    if ((int)(blockIdx.x * 256) >= J.n) return;
    for (int t = threadIdx.x; t < L * L; t += 256) {
        const int j = t / L, k = t - j * L;
        const int lo = j < k ? j : k, hi = j < k ? k : j;
        if (blockIdx.x == 0) W.hop[t] = J.V[(((size_t)lo * L + lo) * L + hi) * L + hi];
        pd[t] = j == k ? 0.0
                       : 2.0 * J.V[(((size_t)j * L + k) * L + j) * L + k] - J.V[(((size_t)j * L + k) * L + k) * L + j];
    }
    for (int t = threadIdx.x; t < L; t += 256)
        d1[t] = 2.0 * J.h[t * L + t] + J.V[(((size_t)t * L + t) * L + t) * L + t];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *J.done = kBatchRunning;
        W.al[kMaxSteps] = W.al[kMaxSteps + 1] = 1e300;  // no test yet
        if (blockIdx.y == 0) *left = 0;
    }
    __syncthreads();
    const int r = blockIdx.x * 256 + threadIdx.x;
    if (r >= J.n) return;
    const str_t s = J.s[r];
    double e = 0.0;
    for (str_t u = s; u; u &= u - 1) {
        const int i = __builtin_ctzll(u);
        e += d1[i];
        for (str_t v = s; v; v &= v - 1) e += pd[i * L + __builtin_ctzll(v)];
    }
    W.dg[r] = e;
}

// Step j of every request: workgroups [0, nchunk) form v_j and H v_j on their
// rows, workgroup nchunk tests T_{j-1}.  NT threads, rows tid + k NT of the
// sums for k < R (n <= NT R).  Dynamic LDS: v_j and the hop elements.
template <int NT, int R>
__global__ void __launch_bounds__(NT) k_doci_batch_step(const DociBatchJob* __restrict__ jobs, int j, int nchunk,
                                                        int count, int* left, int* flag) {
    extern __shared__ __align__(16) unsigned char smem_batch[];
    __shared__ double red[NT / 64];
    const DociBatchJob& J = jobs[blockIdx.y];
    // Finished in an earlier launch.  This launch's test may store j meanwhile, which
    // counts as not finished: the whole workgroup decides alike, and barriers follow.
    if (__hip_atomic_load(J.done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < j) return;
    const int maxs = J.max_steps < kMaxSteps ? J.max_steps : kMaxSteps;
    if ((int)blockIdx.x == nchunk) {
        if (j >= 2 && j - 1 <= maxs) lanczos_test(J, j, maxs, *(TestMatrix*)smem_batch, count, left, flag);
        return;
    }
    const int n = J.n, L = J.L, tid = threadIdx.x;
    const int rows = ((n + nchunk - 1) / nchunk + 63) / 64 * 64, r0 = (int)blockIdx.x * rows;
    if (j > maxs || r0 >= n) return;
    const Work W(J);
    double* x = (double*)smem_batch;
    double* hop = x + n;
    for (int t = tid; t < L * L; t += NT) hop[t] = W.hop[t];
    double w[R];
    double part = 0.0;
    if (j == 0) {
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int r = tid + k * NT;
            w[k] = r < n ? start_value(J.seed, (uint64_t)r) : 0.0;
            part += w[k] * w[k];
        }
    } else {
        const double* u = W.u + (size_t)((j - 1) & 1) * n;
        const double* v = W.v + (size_t)((j + 2) % 3) * n;
        const double* vp = W.v + (size_t)((j + 1) % 3) * n;
        double vj[R];
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int r = tid + k * NT;
            w[k] = r < n ? u[r] : 0.0;
            vj[k] = r < n ? v[r] : 0.0;
        }
        double vq[R];
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int r = tid + k * NT;
            vq[k] = j > 1 && r < n ? vp[r] : 0.0;
        }
        const double beta_prev = j > 1 ? W.be[j - 2] : 0.0;
        double pa = 0.0;
#pragma unroll
        for (int k = 0; k < R; ++k) pa += vj[k] * w[k];
        const double alpha = block_sum<NT>(pa, red);
#pragma unroll
        for (int k = 0; k < R; ++k) {
            w[k] = w[k] - alpha * vj[k] - beta_prev * vq[k];
            part += w[k] * w[k];
        }
        if (blockIdx.x == 0 && tid == 0) W.al[j - 1] = alpha;
    }
    const double beta = sqrt(block_sum<NT>(part, red));
    if (j > 0 && blockIdx.x == 0 && tid == 0) W.be[j - 1] = beta;
    if (j == maxs) return;  // T_maxs is complete
    const double inv = 1.0 / beta;
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int r = tid + k * NT;
        if (r < n) x[r] = w[k] * inv;
    }
    __syncthreads();
    double* vout = W.v + (size_t)(j % 3) * n;
    double* uout = W.u + (size_t)(j & 1) * n;
    const int nh = J.np * J.nv;
    const unsigned char* xb = (const unsigned char*)x;
    const unsigned char* hb = (const unsigned char*)hop;
    const int re = r0 + rows < n ? r0 + rows : n;
    for (int r = r0 + tid; r < re; r += NT) {
        const double xr = x[r];
        vout[r] = xr;
        double acc = W.dg[r] * xr;
        const uint32_t* cp = J.hops + r;
        int t = 0;
        for (; t + 8 <= nh; t += 8) {
            uint32_t e[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) e[q] = cp[(size_t)(t + q) * n];
#pragma unroll
            for (int q = 0; q < 8; ++q)
                acc = fma(*(const double*)(hb + (e[q] >> 17)), *(const double*)(xb + (e[q] & 0x1ffffu)), acc);
        }
        for (; t < nh; ++t) {
            const uint32_t e = cp[(size_t)t * n];
            acc = fma(*(const double*)(hb + (e >> 17)), *(const double*)(xb + (e & 0x1ffffu)), acc);
        }
        uout[r] = acc;
    }
}

int doci_batch_capacity() { return 1024 * 13; }

namespace {
template <int NT, int R>
void run_class(const DociBatchJob* d_jobs, int count, int max_n, int max_L, int max_steps, int* left,
               volatile int* flag, hipEvent_t ev[2], hipStream_t s) {
    const size_t lds = std::max(((size_t)max_n + (size_t)max_L * max_L) * sizeof(double), sizeof(TestMatrix));
    CF_HIP(hipFuncSetAttribute((const void*)k_doci_batch_step<NT, R>, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)lds));
    // enough workgroups to fill the GPU, none with less than a row a thread
    const int nchunk = std::max(1, std::min((max_n + NT - 1) / NT, (1024 + count - 1) / count));
    int* dflag = nullptr;
    CF_HIP(hipHostGetDevicePointer((void**)&dflag, const_cast<int*>(flag), 0));
    // what is queued writes `flag` and the requests' scratch: the caller reads the
    // results and reuses both, also after a launch that throws, only when it has run
    struct Drain {
        hipStream_t s;
        ~Drain() { (void)hipStreamSynchronize(s); }
    } drain{s};
    *flag = 0;
    k_doci_batch_init<<<dim3((unsigned)((max_n + 255) / 256), (unsigned)count), 256, 0, s>>>(d_jobs, left);
    CF_HIP(hipGetLastError());
    constexpr int kAhead = 8;
    const int last = max_steps + 2;  // launches 0 .. max_steps + 1
    for (int j = 0, g = 0; j < last; ++g) {
        for (int e = std::min(last, j + kAhead); j < e; ++j) {
            k_doci_batch_step<NT, R><<<dim3((unsigned)nchunk + 1, (unsigned)count), NT, lds, s>>>(
                d_jobs, j, nchunk, count, left, dflag);
            CF_HIP(hipGetLastError());
        }
        CF_HIP(hipEventRecord(ev[g & 1], s));
        if (g > 0) {
            CF_HIP(hipEventSynchronize(ev[(g - 1) & 1]));
            if (*flag) break;
        }
    }
    CF_HIP(hipStreamSynchronize(s));
}
}  // namespace

void run_doci_batch(const DociBatchJob* d_jobs, int count, int max_n, int max_L, int max_steps, int* left,
                    volatile int* flag, hipEvent_t ev[2], hipStream_t s) {
    if (max_n > 1024 * 13) throw Error(ERR_UNSUPPORTED, "batched DOCI solve: more than 13,312 determinants");
    // requests are grid rows: the device states 65,536 of them, so larger batches run
    // in parts (each request's sums are its own, so its result is the same)
    constexpr int kMost = 32768;
    for (int a = 0; a < count; a += kMost) {
        const int k = std::min(kMost, count - a);
        if (max_n <= 1024) run_class<256, 4>(d_jobs + a, k, max_n, max_L, max_steps, left, flag, ev, s);
        else if (max_n <= 4096) run_class<512, 8>(d_jobs + a, k, max_n, max_L, max_steps, left, flag, ev, s);
        else run_class<1024, 13>(d_jobs + a, k, max_n, max_L, max_steps, left, flag, ev, s);
    }
}

}  // namespace cf
