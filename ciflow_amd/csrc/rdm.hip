// 1- and 2-RDMs as reductions over the string excitation lists.
//
// The reference walks determinant pairs: DensFCI::construct_CI_two_dens is an
// O(n^2/2) pair loop with a popcount classification per pair
// (CIDens.cpp:1582-1631, 855-881), DensDOCI loops over pair hops
// (:1165-1224).  Here:
//
// FCI.  For every determinant K and spin s the one-particle transition
// densities X^s_ab(K) = <K| a+_as a_bs |Psi> are gathered from the single-
// excitation lists of K's strings (diagonal: n_a(K) c_K; a != b: the single
// a -> b of K's s-string, with its phase, times c of the target).  Then
//   gamma^s_ps              = sum_K c_K X^s_ps(K)
//   Gamma^{ab}(pq,rs)       = sum_K X^a_rp(K) X^b_qs(K)
//   Gamma^{ss}(pq,rs)       = sum_K X^s_rp(K) X^s_qs(K) - delta_qr gamma^s_ps
// (from a+_p a+_q a_s a_r = E_pr E_qs - delta_qr E_ps, and for opposite spins
// a+_pa a+_qb a_sb a_ra = E^a_pr E^b_qs), i.e. three Gram products X^T X
// reduced over K in fixed-order chunks (deterministic).
//
// DOCI.  gamma_jj = sum_I c_I^2 n_j(I); D_jk = sum_I c_I^2 n_j n_k;
// P_jk = sum_{J: k in J, j not in J} c_{J-k+j} c_J; each thread owns one (j,k)
// bin and reduces over a chunk of determinants, chunks summed in order.
#include "rdm.h"
#include "string_ops.h"

#include <hipcub/hipcub.hpp>
#include <algorithm>

#include <vector>

namespace cf {

// X^a and X^b rows of determinant K (row-major n x L^2).  Rows must be zeroed.
__global__ void k_build_x(uint64_t da, uint64_t db, int L, const str_t* __restrict__ sa, const str_t* __restrict__ sb,
                          const Exc* __restrict__ suba, const Exc* __restrict__ subb, int Sa, int Sb,
                          const double* __restrict__ c, double* __restrict__ Xa, double* __restrict__ Xb) {
    const uint64_t K = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (K >= da * db) return;
    const uint64_t ka = K / db, kb = K - ka * db;
    const size_t P = (size_t)L * L;
    double* xa = Xa + K * P;
    double* xb = Xb + K * P;
    const double cK = c[K];
    for (str_t s = sa[ka]; s; s &= s - 1) {
        int a = __builtin_ctzll(s);
        xa[a * L + a] = cK;
    }
    for (str_t s = sb[kb]; s; s &= s - 1) {
        int a = __builtin_ctzll(s);
        xb[a * L + a] = cK;
    }
    const Exc* la = suba + ka * (uint64_t)Sa;
    for (int e = 0; e < Sa; ++e) {
        const Exc x = la[e];
        if (x.type != 1) continue;
        double v = c[(uint64_t)x.J * db + kb];
        xa[x.f * L + x.t] = x.sign < 0 ? -v : v;
    }
    const Exc* lb = subb + kb * (uint64_t)Sb;
    for (int e = 0; e < Sb; ++e) {
        const Exc x = lb[e];
        if (x.type != 1) continue;
        double v = c[ka * db + x.J];
        xb[x.f * L + x.t] = x.sign < 0 ? -v : v;
    }
}

// part[chunk][p] = sum_{K in chunk} c_K X[K][p]
__global__ void k_gamma_part(uint64_t n, int P, const double* __restrict__ c, const double* __restrict__ X,
                             uint64_t rows, double* __restrict__ part) {
    const uint64_t k0 = (uint64_t)blockIdx.x * rows;
    uint64_t k1 = k0 + rows;
    if (k1 > n) k1 = n;
    for (int p = threadIdx.x; p < P; p += blockDim.x) {
        double acc = 0.0;
        for (uint64_t K = k0; K < k1; ++K) acc += c[K] * X[K * P + p];
        part[(uint64_t)blockIdx.x * P + p] = acc;
    }
}

// Split-K Gram product: part[chunk][p][q] = sum_{K in chunk} A[K][p] B[K][q].
constexpr int kGT = 32;  // output tile
constexpr int kGK = 32;  // K rows per LDS stage
__global__ void __launch_bounds__(256) k_gram(uint64_t n, int P, const double* __restrict__ A,
                                              const double* __restrict__ B, uint64_t rows, double* __restrict__ part) {
    __shared__ double As[kGK][kGT + 1];
    __shared__ double Bs[kGK][kGT + 1];
    const int nt = (P + kGT - 1) / kGT;
    const int tp = blockIdx.y / nt, tq = blockIdx.y % nt;
    const int p0 = tp * kGT, q0 = tq * kGT;
    const int ty = threadIdx.x / 16, tx = threadIdx.x % 16;
    const uint64_t k0 = (uint64_t)blockIdx.x * rows;
    uint64_t k1 = k0 + rows;
    if (k1 > n) k1 = n;
    double acc00 = 0, acc01 = 0, acc10 = 0, acc11 = 0;
    for (uint64_t kb = k0; kb < k1; kb += kGK) {
        for (int i = threadIdx.x; i < kGK * kGT; i += 256) {
            const int kk = i / kGT, pp = i % kGT;
            const uint64_t K = kb + kk;
            const bool ok = K < k1;
            As[kk][pp] = (ok && p0 + pp < P) ? A[K * P + p0 + pp] : 0.0;
            Bs[kk][pp] = (ok && q0 + pp < P) ? B[K * P + q0 + pp] : 0.0;
        }
        __syncthreads();
#pragma unroll 8
        for (int kk = 0; kk < kGK; ++kk) {
            const double a0 = As[kk][ty * 2], a1 = As[kk][ty * 2 + 1];
            const double b0 = Bs[kk][tx * 2], b1 = Bs[kk][tx * 2 + 1];
            acc00 += a0 * b0;
            acc01 += a0 * b1;
            acc10 += a1 * b0;
            acc11 += a1 * b1;
        }
        __syncthreads();
    }
    const int p = p0 + ty * 2, q = q0 + tx * 2;
    double* o = part + (uint64_t)blockIdx.x * P * P;
    if (p < P && q < P) o[p * P + q] = acc00;
    if (p < P && q + 1 < P) o[p * P + q + 1] = acc01;
    if (p + 1 < P && q < P) o[(p + 1) * P + q] = acc10;
    if (p + 1 < P && q + 1 < P) o[(p + 1) * P + q + 1] = acc11;
}

// The same split-K Gram product on FP64 MFMA (v_mfma_f64_16x16x4f64), for
// P = L^2 <= 256.  A workgroup of 16 wavefronts owns the P x P output of its
// chunk of K rows (or one of `gridDim.y` interleaved parts of it, so that a
// wavefront holds at most TPW = 8 accumulator tiles): 32 rows of A and B are
// staged in LDS per step and every wavefront accumulates its 16 x 16 output
// tiles (tile = 16 (y + gridDim.y t) + wave), so each element of A and B is
// read from HBM gridDim.y times per product.
// 2 n P^2 flop per product.
typedef double v4d __attribute__((ext_vector_type(4)));
constexpr int kGramRows = 32;

template <int TPW>
__global__ void __launch_bounds__(1024) k_gram_mfma(uint64_t n, int P, const double* __restrict__ A,
                                                    const double* __restrict__ B, uint64_t rows,
                                                    double* __restrict__ part) {
    extern __shared__ double gsm[];
    const int SP = P + 1;
    double* As = gsm;
    double* Bs = gsm + kGramRows * SP;
    const int T16 = (P + 15) / 16, ntiles = T16 * T16;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int r = lane & 15, kq = lane >> 4;
    v4d acc[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t) acc[t] = v4d{0.0, 0.0, 0.0, 0.0};
    const uint64_t k0 = (uint64_t)blockIdx.x * rows;
    uint64_t k1 = k0 + rows;
    if (k1 > n) k1 = n;
    for (uint64_t kb = k0; kb < k1; kb += kGramRows) {
        for (int i = threadIdx.x; i < kGramRows * P; i += 1024) {
            const int kk = i / P, pp = i - kk * P;
            const uint64_t K = kb + kk;
            const bool ok = K < k1;
            As[kk * SP + pp] = ok ? A[K * P + pp] : 0.0;
            Bs[kk * SP + pp] = ok ? B[K * P + pp] : 0.0;
        }
        __syncthreads();
        for (int ks = 0; ks < kGramRows; ks += 4) {
            const double* ar = As + (ks + kq) * SP;
            const double* br = Bs + (ks + kq) * SP;
#pragma unroll
            for (int t = 0; t < TPW; ++t) {
                const int tile = 16 * ((int)blockIdx.y + (int)gridDim.y * t) + wave;
                if (tile < ntiles) {
                    const int ti = tile / T16, tj = tile - ti * T16;
                    const int p = ti * 16 + r, q = tj * 16 + r;
                    const double av = p < P ? ar[p] : 0.0;  // A^T[p][K]
                    const double bv = q < P ? br[q] : 0.0;  // B[K][q]
                    acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, acc[t], 0, 0, 0);
                }
            }
        }
        __syncthreads();
    }
    double* o = part + (uint64_t)blockIdx.x * P * P;
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
        const int tile = 16 * ((int)blockIdx.y + (int)gridDim.y * t) + wave;
        if (tile < ntiles) {
            const int ti = tile / T16, tj = tile - ti * T16;
#pragma unroll
            for (int v = 0; v < 4; ++v) {  // D[i][j]: lane j + 16 (i % 4), element i / 4
                const int p = ti * 16 + 4 * v + kq, q = tj * 16 + r;
                if (p < P && q < P) o[(uint64_t)p * P + q] = acc[t][v];
            }
        }
    }
}

// part[chunk] = A^T B over the chunk's rows; MFMA for P <= 256, else k_gram.
static void launch_gram(uint64_t n, int P, const double* A, const double* B, uint64_t rows, uint64_t nchunk,
                        double* part, hipStream_t stream) {
    if (P <= 256) {
        const int T16 = (P + 15) / 16, per = (T16 * T16 + 15) / 16;
        const int split = (per + 7) / 8;  // parts of the output per chunk
        const int tpw = (per + split - 1) / split;
        const size_t lds = 2 * (size_t)kGramRows * (P + 1) * sizeof(double);
        const dim3 grid((unsigned)nchunk, (unsigned)split);
#define CF_GRAM(T) k_gram_mfma<T><<<grid, 1024, lds, stream>>>(n, P, A, B, rows, part)
        if (tpw <= 1) CF_GRAM(1);
        else if (tpw <= 2) CF_GRAM(2);
        else if (tpw <= 4) CF_GRAM(4);
        else CF_GRAM(8);
#undef CF_GRAM
    } else {
        const int nt = (P + kGT - 1) / kGT;
        dim3 grid((unsigned)nchunk, (unsigned)(nt * nt));
        k_gram<<<grid, 256, 0, stream>>>(n, P, A, B, rows, part);
    }
    CF_HIP(hipGetLastError());
}

// out[i] = sum_chunk part[chunk][i]
__global__ void k_sum_chunks(int nchunk, uint64_t len, const double* __restrict__ part, double* __restrict__ out) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= len) return;
    double s = 0.0;
#pragma unroll 8
    for (int c = 0; c < nchunk; ++c) s += part[(uint64_t)c * len + i];
    out[i] = s;
}

// DOCI bins.  part layout per chunk: [0, L^2) D, [L^2, 2L^2) P, [2L^2, 2L^2+L) gamma.
__global__ void k_doci_rdm(uint64_t d, int L, const str_t* __restrict__ s, const uint64_t* __restrict__ binom,
                           const double* __restrict__ c, uint64_t rows, bool two, double* __restrict__ part) {
    const uint64_t i0 = (uint64_t)blockIdx.x * rows;
    uint64_t i1 = i0 + rows;
    if (i1 > d) i1 = d;
    const int L2 = L * L;
    double* o = part + (uint64_t)blockIdx.x * (2 * L2 + L);
    for (int bin = threadIdx.x; bin < L2; bin += blockDim.x) {
        const int j = bin / L, k = bin % L;
        double D = 0.0, Pj = 0.0;
        for (uint64_t I = i0; I < i1; ++I) {
            const str_t x = s[I];
            const bool hj = (x >> j) & 1, hk = (x >> k) & 1;
            const double cI = c[I];
            if (hj && hk) D += cI * cI;
            if (two && j != k && hk && !hj) {
                // J = x holds k, the partner I' = x - k + j holds j
                const str_t y = x ^ ((str_t)1 << k) ^ ((str_t)1 << j);
                Pj += c[rank_bits(y, binom)] * cI;
            }
        }
        o[bin] = D;
        o[L2 + bin] = Pj;
        if (j == k) o[2 * L2 + j] = D;
    }
}

__global__ void __launch_bounds__(256) k_zero(uint64_t n, double* __restrict__ out) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = 0.0;
}

// Gamma[b][p][q][r][t] from the Gram blocks aa, ab, bb ([rp][qt]).
static void unpack_gram(int L, const double* const blocks[3], const double* gamma, double* Gamma) {
    const int P = L * L;
    const size_t L4 = (size_t)P * P;
    for (int b = 0; b < 3; ++b) {
        const double* Gb = blocks[b];
        const int s = b == 2 ? 1 : 0;
        for (int p = 0; p < L; ++p)
            for (int q = 0; q < L; ++q)
                for (int r = 0; r < L; ++r)
                    for (int t = 0; t < L; ++t) {
                        double v = Gb[(size_t)(r * L + p) * P + (q * L + t)];
                        if (b != 1 && q == r) v -= gamma[s * P + p * L + t];
                        Gamma[b * L4 + (((size_t)p * L + q) * L + r) * L + t] = v;
                    }
    }
}

// gamma and Gamma from the transition densities X^a, X^b (n x L^2 rows) and
// the coefficients c_K of the same n determinants (0 for a determinant
// outside the CI space): gamma^s = sum_K c_K X^s(K), Gamma = X^T X Gram
// products minus the contraction term, chunks reduced in fixed order.
static void rdm_from_x(hipStream_t stream, int L, uint64_t n, const double* c, const double* Xa, const double* Xb,
                       double* gamma, double* Gamma) {
    const int P = L * L;
    uint64_t nchunk = (n + 1023) / 1024;
    if (nchunk > 512) nchunk = 512;
    if (nchunk < 1) nchunk = 1;
    const uint64_t rows = (n + nchunk - 1) / nchunk;
    {
        DBuf<double> part(nchunk * (uint64_t)P), tot(2 * (uint64_t)P);
        for (int s = 0; s < 2; ++s) {
            k_gamma_part<<<(unsigned)nchunk, 256, 0, stream>>>(n, P, c, s == 0 ? Xa : Xb, rows, part.p);
            CF_HIP(hipGetLastError());
            k_sum_chunks<<<(unsigned)((P + 255) / 256), 256, 0, stream>>>((int)nchunk, P, part.p, tot.p + s * P);
            CF_HIP(hipGetLastError());
        }
        CF_HIP(hipMemcpyAsync(gamma, tot.p, 2 * P * sizeof(double), hipMemcpyDeviceToHost, stream));
        CF_HIP(hipStreamSynchronize(stream));
    }
    if (!Gamma) return;
    const uint64_t PP = (uint64_t)P * P;
    DBuf<double> part(nchunk * PP), G(3 * PP);
    const double* ops[3][2] = {{Xa, Xa}, {Xa, Xb}, {Xb, Xb}};
    for (int b = 0; b < 3; ++b) {
        launch_gram(n, P, ops[b][0], ops[b][1], rows, nchunk, part.p, stream);
        k_sum_chunks<<<(unsigned)((PP + 255) / 256), 256, 0, stream>>>((int)nchunk, PP, part.p, G.p + b * PP);
        CF_HIP(hipGetLastError());
    }
    std::vector<double> hG(3 * PP);
    CF_HIP(hipMemcpyAsync(hG.data(), G.p, 3 * PP * sizeof(double), hipMemcpyDeviceToHost, stream));
    CF_HIP(hipStreamSynchronize(stream));
    const double* blocks[3] = {hG.data(), hG.data() + PP, hG.data() + 2 * PP};
    unpack_gram(L, blocks, gamma, Gamma);
}

// ---------------------------------------------------------------------------
// FCI densities from one-spin matrices (L <= 16).
//
// For a fixed alpha string ka the transition densities X^a(ka, kb)_rp = s
// c(J, kb) are rows of C with the string J = ka - r + p and the same for every
// kb, so the same-spin part needs no Gram product over determinants: with
//   M^a = C C^T (alpha strings),  M^b = C^T C (beta strings)
//   gamma^a_rp         = sum_ka s M^a(ka, J_rp)
//   sum_K X^a_rp X^a_qs = sum_ka s s' M^a(J_rp, J_qs),
// 2 d^2 (d' ) flop and a gather instead of 2 n L^4.  The opposite-spin part
//   sum_kb X^a_rp(ka, kb) X^b_qs(ka, kb)
// is, per ka, a product of the na (L - na + 1) rows of C that X^a has (of L^2)
// with X^b(ka, .), which is scattered into LDS from C's row ka: 24 instead of 64
// MFMA tiles a step at L=11, nothing stored but each ka's block.  Blocks are
// summed over ka in order.
//
// FCI L=11 5a5b (213,444 determinants): the L^2 columns of X built in memory
// (0.24 + 0.06 ms), three Gram products over them (0.53 ms each) and two
// weighted sums (0.42 ms each) took 3.2 ms a call; now 0.47 ms, of which
// k_gram_ab 0.19 (2.6 GFLOP with the padding, 14 TFLOP/s: the scatter into LDS and
// its barriers), the one-spin matrices 0.03 and the vector's way to the GPU 0.1.
// ---------------------------------------------------------------------------
struct RdmList {   // one nonzero column of X for a string
    uint32_t J;    // string it takes c from
    int16_t ab;    // column r L + p
    int16_t sign;
};

// lists[k][nl]: number operators (J = k), then singles; slot[k][P]: index in
// the list or -1.
__global__ void __launch_bounds__(256) k_rdm_lists(uint64_t d, int L, int nel, int S, const str_t* __restrict__ s,
                                                   const Exc* __restrict__ sub, RdmList* __restrict__ lists,
                                                   int16_t* __restrict__ slot) {
    const uint64_t k = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= d) return;
    const int P = L * L, nl = nel + S - 1;
    RdmList* o = lists + k * (uint64_t)nl;
    int16_t* sl = slot + k * (uint64_t)P;
    for (int p = 0; p < P; ++p) sl[p] = -1;
    int e = 0;
    for (str_t t = s[k]; t; t &= t - 1) {
        const int a = __builtin_ctzll(t);
        o[e] = RdmList{(uint32_t)k, (int16_t)(a * (L + 1)), 1};
        sl[a * (L + 1)] = (int16_t)e++;
    }
    const Exc* x = sub + k * (uint64_t)S;
    for (int i = 0; i < S; ++i)
        if (x[i].type == 1) {
            const int ab = x[i].f * L + x[i].t;
            o[e] = RdmList{x[i].J, (int16_t)ab, (int16_t)(x[i].sign < 0 ? -1 : 1)};
            sl[ab] = (int16_t)e++;
        }
}

// part[z] = partial C C^T (COLS false: rows of the d x m matrix C) or C^T C
// (COLS true: columns of the m x d matrix C) over the z-th part of the m
// dimension; 64 x 64 output blocks, four wavefronts of 2 x 2 MFMA tiles, lower
// block triangle mirrored.
constexpr int kMK = 32;
template <bool COLS>
__global__ void __launch_bounds__(256) k_string_gram(uint64_t d, uint64_t m, uint64_t per,
                                                     const double* __restrict__ C, double* __restrict__ part) {
    __shared__ double As[64][kMK + 1], Bs[64][kMK + 1];
    if (blockIdx.y > blockIdx.x) return;
    const uint64_t i0 = (uint64_t)blockIdx.x * 64, j0 = (uint64_t)blockIdx.y * 64;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int r = lane & 15, kq = lane >> 4, wi = (w >> 1) * 32, wj = (w & 1) * 32;
    const uint64_t k0 = blockIdx.z * per, k1 = k0 + per < m ? k0 + per : m;
    v4d acc[2][2];
    for (int a = 0; a < 2; ++a)
        for (int b = 0; b < 2; ++b) acc[a][b] = v4d{0.0, 0.0, 0.0, 0.0};
    for (uint64_t kb = k0; kb < k1; kb += kMK) {
        double a[8], b[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int t = tid + 256 * q;
            const int x = COLS ? t & 63 : t / kMK, k = COLS ? t >> 6 : t % kMK;
            const bool in = kb + k < k1;
            const uint64_t K = kb + k;
            a[q] = in && i0 + x < d ? C[COLS ? K * d + i0 + x : (i0 + x) * m + K] : 0.0;
            b[q] = in && j0 + x < d ? C[COLS ? K * d + j0 + x : (j0 + x) * m + K] : 0.0;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int t = tid + 256 * q;
            const int x = COLS ? t & 63 : t / kMK, k = COLS ? t >> 6 : t % kMK;
            As[x][k] = a[q];
            Bs[x][k] = b[q];
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < kMK; ks += 4) {
            double av[2], bv[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                av[t] = As[wi + t * 16 + r][ks + kq];
                bv[t] = Bs[wj + t * 16 + r][ks + kq];
            }
#pragma unroll
            for (int ti = 0; ti < 2; ++ti)
#pragma unroll
                for (int tj = 0; tj < 2; ++tj)
                    acc[ti][tj] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[ti], bv[tj], acc[ti][tj], 0, 0, 0);
        }
    }
    double* o = part + blockIdx.z * d * d;
#pragma unroll
    for (int ti = 0; ti < 2; ++ti)
#pragma unroll
        for (int tj = 0; tj < 2; ++tj)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const uint64_t i = i0 + wi + ti * 16 + 4 * v + kq, j = j0 + wj + tj * 16 + r;
                if (i < d && j < d) {
                    o[i * d + j] = acc[ti][tj][v];
                    if (blockIdx.y != blockIdx.x) o[j * d + i] = acc[ti][tj][v];
                }
            }
}

// part[z][rp][qs] over the z-th part of the strings: s s' M(J_rp, J_qs); row P
// of the output is gamma: s M(k, J_qs).  Elements from `first` on.
__global__ void __launch_bounds__(256) k_same_spin_2rdm(uint64_t d, int P, int nl, uint64_t per, int first,
                                                        const RdmList* __restrict__ lists,
                                                        const int16_t* __restrict__ slot, const double* __restrict__ M,
                                                        double* __restrict__ part) {
    const int t = first + blockIdx.x * 256 + threadIdx.x;
    if (t >= (P + 1) * P) return;
    const int rp = t / P, qs = t - rp * P;
    const uint64_t k0 = blockIdx.y * per, k1 = k0 + per < d ? k0 + per : d;
    double acc = 0.0;
    for (uint64_t k = k0; k < k1; ++k) {
        const int e2 = slot[k * P + qs], e1 = rp < P ? slot[k * P + rp] : 0;
        if (e1 < 0 || e2 < 0) continue;
        const RdmList y = lists[k * nl + e2];
        const RdmList x = rp < P ? lists[k * nl + e1] : RdmList{(uint32_t)k, 0, 1};
        const double v = M[(uint64_t)x.J * d + y.J];
        acc += x.sign == y.sign ? v : -v;
    }
    part[(uint64_t)blockIdx.y * (P + 1) * P + t] = acc;
}

// One alpha string's (or part of its beta range's) opposite-spin block:
// out[e][qs] = sum_kb X^a_e(ka, kb) X^b_qs(ka, kb), e over the string's list.
// TB tiles of 16 columns qs, eight wavefronts; TPW output tiles a wavefront.
constexpr int kAbRows = 32;  // beta strings per LDS stage
template <int TPW>
__global__ void __launch_bounds__(512) k_gram_ab(uint64_t db, int P, int nla, int nlb, uint32_t nsplit,
                                                 const RdmList* __restrict__ la, const RdmList* __restrict__ lb,
                                                 const double* __restrict__ c, double* __restrict__ part) {
    extern __shared__ double smem_ab[];
    const int TA = (nla + 15) / 16, TB = (P + 15) / 16, BS = TB * 16 + 1;
    double* As = smem_ab;                             // [TA * 16][kAbRows + 1]
    double* Bs = As + TA * 16 * (kAbRows + 1);        // [kAbRows][BS]
    const uint64_t ka = blockIdx.x / nsplit;
    const uint32_t sp = blockIdx.x - (uint32_t)(ka * nsplit);
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int r = lane & 15, kq = lane >> 4, ntiles = TA * TB;
    const uint64_t steps = (db + kAbRows - 1) / kAbRows;
    const uint64_t s0 = steps * sp / nsplit, s1 = steps * (sp + 1) / nsplit;
    v4d acc[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t) acc[t] = v4d{0.0, 0.0, 0.0, 0.0};
    const RdmList* l = la + ka * (uint64_t)nla;
    const double* row = c + ka * db;
    for (uint64_t s = s0; s < s1; ++s) {
        const uint64_t kb0 = s * kAbRows;
        __syncthreads();  // the last stage has been read
        for (int i = tid; i < kAbRows * BS; i += 512) Bs[i] = 0.0;
        for (int i = tid; i < TA * 16 * kAbRows; i += 512) {
            const int e = i / kAbRows, k = i - e * kAbRows;
            double v = 0.0;
            if (e < nla && kb0 + k < db) {
                const RdmList x = l[e];
                v = c[(uint64_t)x.J * db + kb0 + k];
                if (x.sign < 0) v = -v;
            }
            As[e * (kAbRows + 1) + k] = v;
        }
        __syncthreads();
        for (int i = tid; i < kAbRows * nlb; i += 512) {
            const int k = i / nlb;
            if (kb0 + k >= db) break;
            const RdmList x = lb[(kb0 + k) * nlb + (i - k * nlb)];
            const double v = row[x.J];
            Bs[k * BS + x.ab] = x.sign < 0 ? -v : v;
        }
        __syncthreads();
#pragma unroll 2
        for (int ks = 0; ks < kAbRows; ks += 4) {
#pragma unroll
            for (int t = 0; t < TPW; ++t) {
                const int tile = w + 8 * t;
                if (tile < ntiles) {
                    const int ti = tile / TB, tj = tile - ti * TB;
                    const double av = As[(ti * 16 + r) * (kAbRows + 1) + ks + kq];
                    const double bv = Bs[(ks + kq) * BS + tj * 16 + r];
                    acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, acc[t], 0, 0, 0);
                }
            }
        }
    }
    double* o = part + ((uint64_t)blockIdx.x * nla) * P;
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
        const int tile = w + 8 * t;
        if (tile < ntiles) {
            const int ti = tile / TB, tj = tile - ti * TB;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int e = ti * 16 + 4 * v + kq, q = tj * 16 + r;
                if (e < nla && q < P) o[(uint64_t)e * P + q] = acc[t][v];
            }
        }
    }
}

// part[z][rp][qs] = the blocks of the z-th part of the alpha strings, in order.
__global__ void __launch_bounds__(256) k_sum_ab(uint64_t da, int P, int nla, uint32_t nsplit, uint64_t per,
                                                const int16_t* __restrict__ slot, const double* __restrict__ blocks,
                                                double* __restrict__ part) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= P * P) return;
    const int rp = t / P, qs = t - rp * P;
    const uint64_t k0 = blockIdx.y * per, k1 = k0 + per < da ? k0 + per : da;
    double acc = 0.0;
    for (uint64_t k = k0; k < k1; ++k) {
        const int e = slot[k * P + rp];
        if (e < 0) continue;
        for (uint32_t s = 0; s < nsplit; ++s) acc += blocks[((k * nsplit + s) * nla + e) * P + qs];
    }
    part[(uint64_t)blockIdx.y * P * P + t] = acc;
}

struct RdmSide {
    DBuf<RdmList> lists;
    DBuf<int16_t> slot;
    int nl = 0;
};

static void make_side(RdmSide& s, uint64_t d, int L, int nel, int S, const str_t* str, const Exc* sub,
                      hipStream_t stream) {
    s.nl = nel + S - 1;
    s.lists.alloc(std::max<uint64_t>(1, d * (uint64_t)s.nl));
    s.slot.alloc(d * (uint64_t)L * L);
    k_rdm_lists<<<(unsigned)((d + 255) / 256), 256, 0, stream>>>(d, L, nel, S, str, sub, s.lists.p, s.slot.p);
    CF_HIP(hipGetLastError());
}

// One-spin matrix M = C C^T or C^T C, then that spin's Gram block (with `two`)
// and, in the last row, gamma into out[(P + 1) P].
static void same_spin(bool cols, uint64_t d, uint64_t m, int P, const RdmSide& s, const double* c, bool two, double* out,
                      hipStream_t stream) {
    const unsigned nb = (unsigned)((d + 63) / 64);
    // parts of the sum that fill the GPU, of at least 64 terms, within 1 GiB
    uint64_t z = std::max<uint64_t>(1, 1024 / ((uint64_t)nb * (nb + 1) / 2));
    z = std::min<uint64_t>({z, (m + 63) / 64, std::max<uint64_t>(1, (1ull << 27) / (d * d))});
    const uint64_t per = ((m + z - 1) / z + kMK - 1) / kMK * kMK;
    DBuf<double> parts(z * d * d), M(z > 1 ? d * d : 0);
    const dim3 grid(nb, nb, (unsigned)z);
    if (cols) k_string_gram<true><<<grid, 256, 0, stream>>>(d, m, per, c, parts.p);
    else k_string_gram<false><<<grid, 256, 0, stream>>>(d, m, per, c, parts.p);
    CF_HIP(hipGetLastError());
    if (z > 1) {
        k_sum_chunks<<<(unsigned)((d * d + 255) / 256), 256, 0, stream>>>((int)z, d * d, parts.p, M.p);
        CF_HIP(hipGetLastError());
    }
    const uint64_t len = (uint64_t)(P + 1) * P;
    const uint64_t y = std::max<uint64_t>(1, std::min<uint64_t>(32, d / 8)), yper = (d + y - 1) / y;
    const uint64_t first = two ? 0 : (uint64_t)P * P;
    DBuf<double> sums(y * len);
    k_same_spin_2rdm<<<dim3((unsigned)((len - first + 255) / 256), (unsigned)y), 256, 0, stream>>>(
        d, P, s.nl, yper, (int)first, s.lists.p, s.slot.p, z > 1 ? M.p : parts.p, sums.p);
    CF_HIP(hipGetLastError());
    // (without `two` the sums of the rows before gamma are of unused memory and not read)
    k_sum_chunks<<<(unsigned)((len + 255) / 256), 256, 0, stream>>>((int)y, len, sums.p, out);
    CF_HIP(hipGetLastError());
}

static void rdm_fci(hipStream_t stream, int L, int na, int nb, uint64_t da, uint64_t db, const str_t* sa, const str_t* sb,
                    const Exc* suba, const Exc* subb, int Sa, int Sb, const double* c, double* gamma, double* Gamma) {
    const int P = L * L;
    const uint64_t PP = (uint64_t)P * P, len = PP + P;
    RdmSide A, Bown;
    make_side(A, da, L, na, Sa, sa, suba, stream);
    const bool same = sa == sb;
    if (!same) make_side(Bown, db, L, nb, Sb, sb, subb, stream);
    const RdmSide& B = same ? A : Bown;
    DBuf<double> G(2 * len + PP);  // aa + gamma_a, bb + gamma_b, ab
    same_spin(false, da, db, P, A, c, Gamma != nullptr, G.p, stream);
    same_spin(true, db, da, P, B, c, Gamma != nullptr, G.p + len, stream);
    if (Gamma) {
        double* gab = G.p + 2 * len;
        if (A.nl == 0 || B.nl == 0) {
            k_zero<<<(unsigned)((PP + 255) / 256), 256, 0, stream>>>(PP, gab);
            CF_HIP(hipGetLastError());
        } else {
            const uint64_t steps = (db + kAbRows - 1) / kAbRows;
            const uint32_t nsplit = (uint32_t)std::min<uint64_t>(steps, std::max<uint64_t>(1, 1024 / da));
            DBuf<double> blocks(da * nsplit * (uint64_t)A.nl * P);
            const int TA = (A.nl + 15) / 16, TB = (P + 15) / 16, tpw = (TA * TB + 7) / 8;
            const size_t lds = (size_t)(TA * 16 * (kAbRows + 1) + kAbRows * (TB * 16 + 1)) * sizeof(double);
            const unsigned grid = (unsigned)(da * nsplit);
#define CF_AB(T)                                                                                                \
    do {                                                                                                        \
        if (lds > 64 * 1024)                                                                                    \
            CF_HIP(hipFuncSetAttribute((const void*)k_gram_ab<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)); \
        k_gram_ab<T><<<grid, 512, lds, stream>>>(db, P, A.nl, B.nl, nsplit, A.lists.p, B.lists.p, c, blocks.p);  \
    } while (0)
            if (tpw <= 1) CF_AB(1);
            else if (tpw <= 3) CF_AB(3);
            else if (tpw <= 6) CF_AB(6);
            else CF_AB(10);
#undef CF_AB
            CF_HIP(hipGetLastError());
            const uint64_t y = std::max<uint64_t>(1, std::min<uint64_t>(32, da / 8)), yper = (da + y - 1) / y;
            DBuf<double> sums(y * PP);
            k_sum_ab<<<dim3((unsigned)((PP + 255) / 256), (unsigned)y), 256, 0, stream>>>(da, P, A.nl, nsplit, yper,
                                                                                     A.slot.p, blocks.p, sums.p);
            CF_HIP(hipGetLastError());
            k_sum_chunks<<<(unsigned)((PP + 255) / 256), 256, 0, stream>>>((int)y, PP, sums.p, gab);
            CF_HIP(hipGetLastError());
        }
    }
    std::vector<double> h(2 * len + PP);
    CF_HIP(hipMemcpyAsync(h.data(), G.p, (Gamma ? 2 * len + PP : 2 * len) * sizeof(double), hipMemcpyDeviceToHost, stream));
    CF_HIP(hipStreamSynchronize(stream));
    for (int s = 0; s < 2; ++s) std::copy_n(h.data() + s * len + PP, P, gamma + s * P);
    if (!Gamma) return;
    const double* blocks3[3] = {h.data(), h.data() + 2 * len, h.data() + len};
    unpack_gram(L, blocks3, gamma, Gamma);
}

void rdm_dense(hipStream_t stream, int kind, int L, int nup, int ndown, uint64_t da, uint64_t db, const str_t* sa,
               const str_t* sb, const Exc* suba, const Exc* subb, int Sa, int Sb, const uint64_t* binom,
               const double* c_host, uint64_t n, double* gamma, double* Gamma) {
    const int P = L * L;
    DBuf<double> c(n);
    CF_HIP(hipMemcpyAsync(c.p, c_host, n * sizeof(double), hipMemcpyHostToDevice, stream));
    std::vector<double> g(2 * (size_t)P, 0.0);
    if (kind == 1) {  // DOCI
        // 16 rows a workgroup while that fills the GPU: each thread's bin is a
        // serial loop over them (252 rows in one workgroup took 151 us).  With the
        // pair bins, whose terms wait for a gather, long loops want twice as many
        // (512 / 1,024 workgroups: L=18 0.37 / 0.36 ms, L=20 0.67 / 0.56, L=22 2.64 /
        // 2.16, L=24 13.4 / 12.1); without them the shorter sum over chunks wins
        // (L=18 0.085 / 0.107 ms, L=20 0.167 / 0.180, L=24 1.47 / 1.45)
        uint64_t nchunk = (n + 15) / 16;
        const uint64_t most = Gamma && n >= 100000 ? 1024 : 512;
        if (nchunk > most) nchunk = most;
        if (nchunk < 1) nchunk = 1;
        const uint64_t rows = (n + nchunk - 1) / nchunk;
        const uint64_t len = 2 * (uint64_t)P + L;
        DBuf<double> part(nchunk * len), tot(len);
        int thr = P < 1024 ? ((P + 63) / 64) * 64 : 1024;
        k_doci_rdm<<<(unsigned)nchunk, thr, 0, stream>>>(n, L, sa, binom, c.p, rows, Gamma != nullptr, part.p);
        CF_HIP(hipGetLastError());
        k_sum_chunks<<<(unsigned)((len + 255) / 256), 256, 0, stream>>>((int)nchunk, len, part.p, tot.p);
        CF_HIP(hipGetLastError());
        std::vector<double> h(len);
        CF_HIP(hipMemcpyAsync(h.data(), tot.p, len * sizeof(double), hipMemcpyDeviceToHost, stream));
        CF_HIP(hipStreamSynchronize(stream));
        for (int j = 0; j < L; ++j) {
            gamma[j * L + j] = h[2 * P + j];
            gamma[P + j * L + j] = h[2 * P + j];
        }
        for (int p = 0; p < L; ++p)
            for (int q = 0; q < L; ++q)
                if (p != q) gamma[p * L + q] = gamma[P + p * L + q] = 0.0;
        if (Gamma) {
            const size_t L4 = (size_t)P * P;
            std::fill(Gamma, Gamma + 3 * L4, 0.0);
            auto at = [&](int b, int i, int j, int k, int l) -> double& {
                return Gamma[b * L4 + (((size_t)i * L + j) * L + k) * L + l];
            };
            for (int j = 0; j < L; ++j)
                for (int k = 0; k < L; ++k) {
                    const double D = h[j * L + k];
                    at(1, j, k, j, k) = D;
                    if (j != k) {
                        at(0, j, k, j, k) = D;
                        at(0, j, k, k, j) = -D;
                        at(2, j, k, j, k) = D;
                        at(2, j, k, k, j) = -D;
                        at(1, j, j, k, k) = h[P + j * L + k];
                    }
                }
        }
        return;
    }
    // FCI up to L = 16 (12,870 strings a spin): one-spin matrices; at most 1.3 GB for
    // one of them and, with the 2-RDM, 1.9 GB of opposite-spin blocks beside the
    // vector.  Above, X in memory, and for the 1-RDM alone of a space with hardly
    // any strings of one spin: X has n L^2 entries then where the matrix has d^2 (one-spin
    // / X, ms: L=16 8a0b d^2 = 50 n L^2 1.29 / 0.61, 6a0b 31 n L^2 0.72 / 0.59, L=15 7a0b 29
    // 0.53 / 0.56, L=14 7a0b 17 0.29 / 0.49, L=16 8a1b 3 1.37 / 1.48)
    const bool narrow = !Gamma && da * da + db * db > 30 * n * (uint64_t)P;
    if (L <= 16 && !narrow) {
        rdm_fci(stream, L, nup, ndown, da, db, sa, sb, suba, subb, Sa, Sb, c.p, gamma, Gamma);
        return;
    }
    DBuf<double> Xa(n * (uint64_t)P), Xb(n * (uint64_t)P);
    CF_HIP(hipMemsetAsync(Xa.p, 0, Xa.bytes(), stream));
    CF_HIP(hipMemsetAsync(Xb.p, 0, Xb.bytes(), stream));
    k_build_x<<<(unsigned)((n + 127) / 128), 128, 0, stream>>>(da, db, L, sa, sb, suba, subb, Sa, Sb, c.p, Xa.p, Xb.p);
    CF_HIP(hipGetLastError());
    rdm_from_x(stream, L, n, c.p, Xa.p, Xb.p, gamma, Gamma);
}

// ---------------------------------------------------------------------------
// Determinant lists (DensFILE, CIDens.cpp:1468-1526).  The same transition
// densities and Gram products as for FCI, over the determinants K that one
// single excitation reaches from the list (the list included): K is keyed
// up | down << L, the keys are sorted and made unique (hipCUB), and every
// list determinant J scatters c_J into X^s[K][a*L + b] for K = J - b + a
// (b occupied in J's s-string, a = b or empty), with the single's phase.
// (K, s, a, b) fixes J, so the scatter has no conflicts and is deterministic.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t det_key(str_t u, str_t d, int L) { return (uint64_t)u | ((uint64_t)d << L); }

// keys[J*E + e]: J itself, then its alpha singles, then its beta singles.
__global__ void k_det_closure_keys(uint64_t n, int L, int E, const str_t* __restrict__ up,
                                   const str_t* __restrict__ down, uint64_t* __restrict__ keys) {
    const uint64_t J = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (J >= n) return;
    const str_t u = up[J], d = down[J];
    const str_t full = L >= 64 ? ~(str_t)0 : (((str_t)1 << L) - 1);
    uint64_t* o = keys + J * (uint64_t)E;
    int e = 0;
    o[e++] = det_key(u, d, L);
    for (str_t t = u; t; t &= t - 1) {
        const str_t bb = t & (~t + 1);
        for (str_t v = full & ~u; v; v &= v - 1) o[e++] = det_key((u ^ bb) | (v & (~v + 1)), d, L);
    }
    for (str_t t = d; t; t &= t - 1) {
        const str_t bb = t & (~t + 1);
        for (str_t v = full & ~d; v; v &= v - 1) o[e++] = det_key(u, (d ^ bb) | (v & (~v + 1)), L);
    }
}

__device__ __forceinline__ uint64_t find_key(const uint64_t* __restrict__ ks, uint64_t nk, uint64_t key) {
    uint64_t lo = 0, hi = nk;  // first index with ks[i] >= key
    while (lo < hi) {
        const uint64_t mid = (lo + hi) >> 1;
        if (ks[mid] < key) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

__global__ void k_det_scatter_x(uint64_t n, int L, const str_t* __restrict__ up, const str_t* __restrict__ down,
                                const double* __restrict__ c, const uint64_t* __restrict__ ks, uint64_t nk,
                                double* __restrict__ cK, double* __restrict__ Xa, double* __restrict__ Xb) {
    const uint64_t J = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (J >= n) return;
    const str_t u = up[J], d = down[J];
    const str_t full = L >= 64 ? ~(str_t)0 : (((str_t)1 << L) - 1);
    const size_t P = (size_t)L * L;
    const double cj = c[J];
    const uint64_t self = find_key(ks, nk, det_key(u, d, L));
    cK[self] = cj;
    for (str_t t = u; t; t &= t - 1) {  // diagonal: X^a[J][b*L + b] = c_J
        const int b = __builtin_ctzll(t);
        Xa[self * P + b * L + b] = cj;
    }
    for (str_t t = d; t; t &= t - 1) {
        const int b = __builtin_ctzll(t);
        Xb[self * P + b * L + b] = cj;
    }
    for (int s = 0; s < 2; ++s) {
        const str_t own = s == 0 ? u : d;
        double* X = s == 0 ? Xa : Xb;
        for (str_t t = own; t; t &= t - 1) {
            const int b = __builtin_ctzll(t);
            for (str_t v = full & ~own; v; v &= v - 1) {
                const int a = __builtin_ctzll(v);
                const str_t ks_ = (own ^ ((str_t)1 << b)) | ((str_t)1 << a);  // K's s-string: J - b + a
                const uint64_t key = s == 0 ? det_key(ks_, d, L) : det_key(u, ks_, L);
                const uint64_t k = find_key(ks, nk, key);
                const int ph = stacked(own & ks_, a, b) & 1;  // <K| a+_a a_b |J> phase
                X[k * P + a * L + b] = ph ? -cj : cj;
            }
        }
    }
}

__global__ void k_count_equal_neighbours(uint64_t n, const uint64_t* __restrict__ k, unsigned int* __restrict__ dup) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i + 1 < n && k[i] == k[i + 1]) atomicAdd(dup, 1u);
}

void rdm_dets(hipStream_t stream, int L, uint64_t n, const str_t* up, const str_t* down, const double* c_host,
              double* gamma, double* Gamma) {
    if (2 * L > 64) throw Error(ERR_UNSUPPORTED, "determinant-list RDMs need L <= 32");
    int na = 0, nb = 0;
    {
        str_t u0 = 0, d0 = 0;
        CF_HIP(hipMemcpyAsync(&u0, up, sizeof(str_t), hipMemcpyDeviceToHost, stream));
        CF_HIP(hipMemcpyAsync(&d0, down, sizeof(str_t), hipMemcpyDeviceToHost, stream));
        CF_HIP(hipStreamSynchronize(stream));
        na = __builtin_popcountll(u0);
        nb = __builtin_popcountll(d0);
    }
    const int E = 1 + na * (L - na) + nb * (L - nb);
    const uint64_t nkeys = n * (uint64_t)E;
    const unsigned grid = (unsigned)((n + 127) / 128);
    DBuf<uint64_t> keys(nkeys), sorted(nkeys), uniq(nkeys);
    DBuf<int> nsel(1);
    k_det_closure_keys<<<grid, 128, 0, stream>>>(n, L, E, up, down, keys.p);
    CF_HIP(hipGetLastError());
    // the list itself must not repeat a determinant (its key sits at keys[J*E])
    {
        DBuf<uint64_t> lk(n), lks(n);
        DBuf<unsigned int> dup(1);
        CF_HIP(hipMemcpy2DAsync(lk.p, sizeof(uint64_t), keys.p, E * sizeof(uint64_t), sizeof(uint64_t), n,
                                hipMemcpyDeviceToDevice, stream));
        size_t tb = 0;
        CF_HIP(hipcub::DeviceRadixSort::SortKeys(nullptr, tb, lk.p, lks.p, (int)n, 0, 2 * L, stream));
        DBuf<char> tmp(tb ? tb : 1);
        CF_HIP(hipcub::DeviceRadixSort::SortKeys(tmp.p, tb, lk.p, lks.p, (int)n, 0, 2 * L, stream));
        CF_HIP(hipMemsetAsync(dup.p, 0, sizeof(unsigned int), stream));
        k_count_equal_neighbours<<<grid, 128, 0, stream>>>(n, lks.p, dup.p);
        CF_HIP(hipGetLastError());
        unsigned int hd = 0;
        CF_HIP(hipMemcpyAsync(&hd, dup.p, sizeof(unsigned int), hipMemcpyDeviceToHost, stream));
        CF_HIP(hipStreamSynchronize(stream));
        if (hd) throw Error(ERR_ARG, "determinant list repeats a determinant; RDMs need distinct determinants");
    }
    if (nkeys > 0x7fffffffull) throw Error(ERR_UNSUPPORTED, "determinant list too long for the RDM closure");
    size_t tb = 0, tb2 = 0;
    CF_HIP(hipcub::DeviceRadixSort::SortKeys(nullptr, tb, keys.p, sorted.p, (int)nkeys, 0, 2 * L, stream));
    CF_HIP(hipcub::DeviceSelect::Unique(nullptr, tb2, sorted.p, uniq.p, nsel.p, (int)nkeys, stream));
    DBuf<char> tmp(std::max(tb, tb2) ? std::max(tb, tb2) : 1);
    CF_HIP(hipcub::DeviceRadixSort::SortKeys(tmp.p, tb, keys.p, sorted.p, (int)nkeys, 0, 2 * L, stream));
    CF_HIP(hipcub::DeviceSelect::Unique(tmp.p, tb2, sorted.p, uniq.p, nsel.p, (int)nkeys, stream));
    int hk = 0;
    CF_HIP(hipMemcpyAsync(&hk, nsel.p, sizeof(int), hipMemcpyDeviceToHost, stream));
    CF_HIP(hipStreamSynchronize(stream));
    const uint64_t nk = (uint64_t)hk;
    const size_t P = (size_t)L * L;
    DBuf<double> c(n), cK(nk), Xa(nk * P), Xb(nk * P);
    CF_HIP(hipMemcpyAsync(c.p, c_host, n * sizeof(double), hipMemcpyHostToDevice, stream));
    CF_HIP(hipMemsetAsync(cK.p, 0, cK.bytes(), stream));
    CF_HIP(hipMemsetAsync(Xa.p, 0, Xa.bytes(), stream));
    CF_HIP(hipMemsetAsync(Xb.p, 0, Xb.bytes(), stream));
    k_det_scatter_x<<<grid, 128, 0, stream>>>(n, L, up, down, c.p, uniq.p, nk, cK.p, Xa.p, Xb.p);
    CF_HIP(hipGetLastError());
    rdm_from_x(stream, L, nk, cK.p, Xa.p, Xb.p, gamma, Gamma);
}

void pack_rdm(int L, const double* gamma, const double* Gamma, double* one, double* two) {
    const size_t osz = (size_t)L * (L + 1) / 2;
    for (int s = 0; s < 2; ++s)
        for (int p = 0; p < L; ++p)
            for (int q = p; q < L; ++q) one[s * osz + (size_t)p * L + q - (size_t)p * (p + 1) / 2] = gamma[s * L * L + p * L + q];
    if (!two || !Gamma) return;
    const size_t C = (size_t)L * L;
    const size_t tsz = C * (C + 1) / 2;
    const size_t L4 = C * C;
    auto idx = [&](size_t r, size_t c) { return C * r + c - r * (r + 1) / 2; };
    for (size_t i = 0; i < 3 * tsz; ++i) two[i] = 0.0;
    for (int i = 0; i < L; ++i)
        for (int j = 0; j < L; ++j)
            for (int k = 0; k < L; ++k)
                for (int l = 0; l < L; ++l) {
                    const size_t P1 = (size_t)i * L + j, Q1 = (size_t)k * L + l;
                    if (P1 <= Q1) two[tsz + idx(P1, Q1)] = Gamma[L4 + (((size_t)i * L + j) * L + k) * L + l];
                    if (i < j && k < l) {
                        const size_t P = (size_t)i * L + j - (size_t)(i + 1) * (i + 2) / 2;
                        const size_t Q = (size_t)k * L + l - (size_t)(k + 1) * (k + 2) / 2;
                        if (P <= Q) {
                            two[idx(P, Q)] = Gamma[(((size_t)i * L + j) * L + k) * L + l];
                            two[2 * tsz + idx(P, Q)] = Gamma[2 * L4 + (((size_t)i * L + j) * L + k) * L + l];
                        }
                    }
                }
}

}  // namespace cf
