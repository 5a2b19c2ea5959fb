// DOCI SpMV on position-major pair-hop columns (replaces SparseMatrix_CRS_Sym::mvprod,
// SparseMatrix_CRS.cpp:700-723, for DOCI matrices built by DOCI::construct_CI_matrix,
// CIMethod.cpp:611-660).
//
// A DOCI row is one pair string s; its off-diagonal elements are the hops of a
// pair from an occupied orbital j to an empty orbital k, with element
// V(m, m, M, M) (m = min(j, k), M = max(j, k)) and phase +1, so the value
// depends on the hop only.  The CRS stores 12 (FP64) or 8 (FP32) bytes per
// element; here a thread per row walks its np * nv hops in a fixed order (a-th
// occupied orbital from the top, b-th empty orbital from the top), takes the
// value from an L x L pair table in LDS and the target rank from a
// position-major column array, col[t * n + i], read as one contiguous
// wavefront load per slot.  Elements the CRS build drops (|v| <= zero) are
// zero in the table, so the product equals the CRS product up to summation
// order.  Rows in rank order share their high orbitals, so a slot's targets
// across a wavefront fall into a few nearby x segments.
//
// HBM-bound.  Algorithmic bytes per call:
//   B = n * (4 * np * nv + 8 (string) + 8 (diagonal) + 8 (x once) + 8 (y)).
#include "spmv_doci.h"
#include "string_ops.h"

#include <type_traits>

namespace cf {

__global__ void __launch_bounds__(256) k_doci_ell_fill(DociEllArgs a, const uint64_t* __restrict__ binom,
                                                       uint32_t* __restrict__ col) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= a.n) return;
    const str_t full = a.L == 64 ? ~0ull : (((str_t)1 << a.L) - 1);
    const str_t s = a.s[i], vir = ~s & full;
    uint64_t t = 0;
    str_t o = s;
    for (int p = 0; p < a.np; ++p) {
        const int j = 63 - __builtin_clzll(o);
        o ^= (str_t)1 << j;
        str_t v = vir;
        for (int q = 0; q < a.nv; ++q) {
            const int k = 63 - __builtin_clzll(v);
            v ^= (str_t)1 << k;
            col[t * a.n + i] = rank_bits(s ^ ((str_t)1 << j) ^ ((str_t)1 << k), binom);
            ++t;
        }
    }
}

void launch_doci_ell_fill(const DociEllArgs& a, const uint64_t* binom, uint32_t* col, hipStream_t s) {
    if (!a.n || !a.np || !a.nv) return;
    k_doci_ell_fill<<<(unsigned)((a.n + 255) / 256), 256, 0, s>>>(a, binom, col);
    CF_HIP(hipGetLastError());
}

__global__ void k_doci_pair_table(int L, HamDev H, double zero, double* __restrict__ vk64,
                                  float* __restrict__ vk32) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= L * L) return;
    const int j = t / L, k = t - j * L;
    const size_t lo = j < k ? j : k, hi = j < k ? k : j;
    double v = H.V[((lo * L + lo) * L + hi) * L + hi];
    if (!(fabs(v) > zero)) v = 0.0;
    vk64[t] = v;
    vk32[t] = (float)v;
}

void launch_doci_pair_table(const DociEllArgs& a, HamDev H, double* vk64, float* vk32, hipStream_t s) {
    const int LL = a.L * a.L;
    k_doci_pair_table<<<(LL + 255) / 256, 256, 0, s>>>(a.L, H, a.zero, vk64, vk32);
    CF_HIP(hipGetLastError());
}

// SUB lanes share a row, lane `sub` taking the occupied orbitals a = sub,
// sub + SUB, ... (small spaces need several lanes per row to fill the GPU);
// U slots per batch: U column loads, then U x gathers, then U FMAs, so each
// lane keeps U independent gathers in flight.
template <typename VT, int SUB, int U>
__global__ void __launch_bounds__(1024) k_spmv_doci(DociEllArgs a, const VT* __restrict__ vk,
                                                    const double* __restrict__ x, double* __restrict__ y) {
    extern __shared__ double smem_doci[];
    VT* tab = reinterpret_cast<VT*>(smem_doci);
    const int L = a.L;
    for (int t = threadIdx.x; t < L * L; t += blockDim.x) tab[t] = vk[t];
    __syncthreads();
    const uint64_t n = a.n;
    const uint64_t i = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / SUB;
    const int sub = (int)(threadIdx.x % SUB);
    const bool live = i < n;
    double acc = 0.0;
    if (live) {
        const str_t full = L == 64 ? ~0ull : (((str_t)1 << L) - 1);
        const str_t s = a.s[i], vir = ~s & full;
        if (sub == 0) {
            double d = a.diag[i];
            if (!(fabs(d) > a.zero)) d = 0.0;
            acc = (double)(VT)d * x[i];
        }
        const int nv = a.nv;
        const uint32_t na = a.np > sub ? (uint32_t)((a.np - sub + SUB - 1) / SUB) : 0u;
        const uint32_t R1 = na * (uint32_t)nv;
        const uint32_t* cp = a.col + i;
        str_t o = s, v = 0;
        for (int q = 0; q < sub && o; ++q) o ^= (str_t)1 << (63 - __builtin_clzll(o));
        int j = 0;
        uint32_t slot = 0;  // a * nv + b of the next hop
        for (uint32_t t0 = 0; t0 < R1; t0 += U) {
            uint32_t c[U];
            double w[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                c[u] = 0;
                w[u] = 0.0;
                if (t0 + u < R1) {
                    if (!v) {  // next occupied orbital of this lane: a += SUB
                        if (t0 + u) {
                            slot += (uint32_t)(SUB - 1) * (uint32_t)nv;
                            for (int q = 1; q < SUB && o; ++q) o ^= (str_t)1 << (63 - __builtin_clzll(o));
                        } else {
                            slot = (uint32_t)sub * (uint32_t)nv;
                        }
                        j = 63 - __builtin_clzll(o);
                        o ^= (str_t)1 << j;
                        v = vir;
                    }
                    const int k = 63 - __builtin_clzll(v);
                    v ^= (str_t)1 << k;
                    w[u] = (double)tab[j * L + k];
                    c[u] = __builtin_nontemporal_load(cp + (uint64_t)slot * n);
                    ++slot;
                }
            }
            double xv[U];
#pragma unroll
            for (int u = 0; u < U; ++u) xv[u] = t0 + u < R1 ? x[c[u]] : 0.0;
#pragma unroll
            for (int u = 0; u < U; ++u) acc += w[u] * xv[u];
        }
    }
#pragma unroll
    for (int off = SUB / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, SUB);
    if (live && sub == 0) y[i] = acc;
}

DociShape doci_default_shape(uint64_t n) {
    // enough lanes for ~2 waves per SIMD on 256 CUs: 131,072 lanes
    DociShape sh;
    sh.threads = 256;
    sh.sub = 1;
    while (sh.sub < 8 && n * (uint64_t)sh.sub < 131072) sh.sub *= 2;
    return sh;
}

template <typename VT>
static void launch_doci(const DociEllArgs& a, DociShape sh, const VT* vk, const double* x, double* y,
                        hipStream_t s) {
    if (!a.n) return;
    const int T = sh.threads;
    const uint64_t lanes = a.n * (uint64_t)sh.sub;
    const uint64_t nb = (lanes + T - 1) / T;
    CF_REQUIRE(nb < (1ull << 31), "too many rows for one DOCI SpMV launch");
    const size_t shm = (size_t)a.L * a.L * sizeof(VT);
    switch (sh.sub) {
        case 1: k_spmv_doci<VT, 1, 8><<<(uint32_t)nb, T, shm, s>>>(a, vk, x, y); break;
        case 2: k_spmv_doci<VT, 2, 8><<<(uint32_t)nb, T, shm, s>>>(a, vk, x, y); break;
        case 4: k_spmv_doci<VT, 4, 8><<<(uint32_t)nb, T, shm, s>>>(a, vk, x, y); break;
        case 8: k_spmv_doci<VT, 8, 8><<<(uint32_t)nb, T, shm, s>>>(a, vk, x, y); break;
        default: CF_REQUIRE(false, "DOCI SpMV: lanes per row must be 1, 2, 4 or 8");
    }
    CF_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Block-staged product: no stored columns.  Rows sharing the high part hi of
// their string form the contiguous rank range base(hi, c) + rank_lo(lo), with
// rank(s) = sum_m C(k_m, m) split at the w-th orbital:
//   base(hi, c) = sum over the high bits (m = c+1, c+2, ...) of C(w + q, m).
// A workgroup owns one block (R = C(w, c) rows, every row with the same c, so
// every loop over its hops has the same trip count in every lane):
//   low -> low hops:   target in the own block, x staged in LDS once;
//   high -> high hops: block (hi ^ jh ^ kh, c), same low pattern, so the same
//                      row index: one coalesced read of the neighbour block;
//   high -> low hops:  block (hi ^ jh, c + 1), staged in LDS per jh;
//   low -> high hops:  block (hi | kh, c - 1), staged in LDS per kh, beside the former.
// Per product the x blocks pass through L2 about 1 + ch (L - w - ch) times
// (ch high pairs) plus the staged blocks; HBM sees x, y and the diagonal once.
// ---------------------------------------------------------------------------
constexpr int kBlkHops = 128;   // high -> high hops per block: ch (nh - ch) <= 100 for nh <= 20
constexpr int kBlkStages = 32;  // staged blocks per block: nh <= 20

// First ranks of the blocks that hops of one high pair reach, from prefix sums.
// Bit q of hi with e bits below it adds C(w + q, c + 1 + e) to base(hi, c).  Taking
// a bit away, adding one or moving one changes e (and c) by one on a contiguous
// range of the other bits, so every such base is a few differences of the prefix
// sums P[s] of C(w + q, c + 1 + e + s) over the set bits, s = -1, 0, 1, and the
// terms E[s][q] of single orbitals.  One load an orbital and shift (a walk over
// the bits of each target was a chain of as many dependent loads).
struct BlockSums {
    uint32_t P[3][33], E[3][32];
    // the first wavefront: lane q holds orbital q
    __device__ __forceinline__ void fill(uint32_t hi, int c, int w, int nh, const uint64_t* __restrict__ binom) {
        const int l = threadIdx.x, q = l & 31;
        const int e = __builtin_popcount(hi & ((1u << q) - 1));
        const bool set = q < nh && ((hi >> q) & 1u);
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            const int m = c + e + s;  // C(n, m) of the rank table: m <= 31 orbitals' pairs
            const uint32_t v = q < nh && m >= 0 ? (uint32_t)binom[(w + q) * kBinomCols + m] : 0u;
            uint32_t p = set ? v : 0u;
#pragma unroll
            for (int o = 1; o < 32; o <<= 1) {
                const uint32_t u = __shfl_up(p, o, 32);
                if (q >= o) p += u;
            }
            if (l < 32) {
                E[s][q] = v;
                P[s][q + 1] = p;
                if (q == 0) P[s][0] = 0;
            }
        }
    }
    // bits a <= q < b with shift s - 1
    __device__ __forceinline__ uint32_t sum(int s, int a, int b) const { return P[s][b] - P[s][a]; }
    // hi without j, one low pair more: bits below j count one more pair under them
    __device__ __forceinline__ uint32_t removed(int j) const { return sum(2, 0, j) + sum(1, j + 1, 32); }
    // hi with k, one low pair less
    __device__ __forceinline__ uint32_t added(int k) const { return sum(0, 0, k) + E[0][k] + sum(1, k, 32); }
    // hi without j and with k, same low pairs
    __device__ __forceinline__ uint32_t moved(int j, int k) const {
        return j < k ? sum(1, 0, j) + sum(0, j + 1, k) + E[0][k] + sum(1, k, 32)
                     : sum(1, 0, k) + E[1][k] + sum(2, k, j) + sum(1, j + 1, 32);
    }
};

// The low pattern of a row fixes the LDS offsets of all its hops, so they come
// from a table (k_doci_hop_table), two 16-bit offsets a word, read coalesced.  A
// hop across the split at low orbital k takes the row l | k of a high -> low stage
// if k is empty in l, the row l ^ k of a low -> high stage if it is occupied: one
// stage of either kind is in LDS at a time (xa, xb) and each row does one hop per
// k.  A hop inside the low part takes pair (j, k) for every row, from a slot of
// zero where both or neither is occupied.  Pair elements are then the same for
// the whole workgroup (scalar registers), the loops over orbitals are unrolled and
// their LDS reads independent.  Walking each row's bits took three dependent LDS
// reads and ten VALU operations a hop, and was latency-bound.  A wavefront without
// rows of the block only stages.  L=23 (11 pairs), n = 1,352,078: 95 -> 81 us; 12
// vectors of L=19 (9 pairs), n = 92,378: 71 -> 46 us.  What is left: LDS and VALU
// are busy 45% and 43% of the time, the rest is waits (a workgroup's stages follow
// each other); blocks sorted by c, 512 threads of one row (90 us) and the table
// words loaded ahead (83) did not help.
struct DociInst {
    int W;         // low orbitals the instance is unrolled for
    uint32_t cap;  // rows of an x block in LDS
};
__host__ __device__ constexpr uint32_t doci_zero_off(uint32_t cap) { return 2 * cap * 8; }
__host__ __device__ constexpr int doci_ll_words(int W) { return (W * (W - 1) / 2 + 1) / 2; }
__host__ __device__ constexpr int doci_words(int W) { return doci_ll_words(W) + (W + 1) / 2; }
static DociInst doci_inst(int w) {
    if (w <= 7) return {7, 64};
    if (w <= 9) return {9, 128};
    if (w <= 10) return {10, 256};
    if (w <= 11) return {11, 512};
    return {12, 1024};
}

// words[d * 2^w + position of low pattern l in lo_of]: offsets of pairs (j, k),
// k < j in order, then of the orbitals k.
__global__ void __launch_bounds__(256) k_doci_hop_table(DociBlockArgs a, DociInst in, uint32_t* __restrict__ words) {
    const uint32_t nlo = 1u << a.w;
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    const int d = blockIdx.y, nll = doci_ll_words(in.W), np = in.W * (in.W - 1) / 2;
    if (i >= nlo) return;
    const uint32_t l = a.lo_of[i];
    uint32_t word = 0;
    for (int e = 0; e < 2; ++e) {
        uint32_t off = doci_zero_off(in.cap);
        if (d < nll) {
            int j = 1, p = 2 * d + e;
            if (p < np) {
                while (p >= j) p -= j++;
                if (j < a.w && (((l >> j) ^ (l >> p)) & 1u)) off = a.rank_lo[l ^ (1u << j) ^ (1u << p)] * 8u;
            }
        } else {
            const int k = 2 * (d - nll) + e;
            if (k < a.w) off = a.rank_lo[l ^ (1u << k)] * 8u + ((l >> k) & 1u ? in.cap * 8u : 0u);
        }
        word |= off << (16 * e);
    }
    words[(size_t)d * nlo + i] = word;
}

size_t doci_hop_words(int w) { return (size_t)doci_words(doci_inst(w).W) << w; }

void launch_doci_hop_table(const DociBlockArgs& a, uint32_t* words, hipStream_t s) {
    CF_REQUIRE(a.w >= 1 && a.w <= kDociMaxW, "block-staged DOCI SpMV: 1 <= w <= 12 low orbitals");
    const DociInst in = doci_inst(a.w);
    k_doci_hop_table<<<dim3(((1u << a.w) + 255) / 256, (unsigned)doci_words(in.W)), 256, 0, s>>>(a, in, words);
    CF_HIP(hipGetLastError());
}

// The pair table through scalar loads: read-only while the kernel runs, uniform
// indices (a batch lane's table pointer comes from memory, so without the
// constant address space its reads were flat loads, which wait on LDS too).
template <typename VT>
using PairTab = const __attribute__((address_space(4))) VT*;

__device__ __forceinline__ double at_byte(const double* base, uint32_t off) {
    return *(const double*)((const char*)base + off);
}

// Hops inside the low part for Q rows a lane; hop[q]: the row's first table word.
template <typename VT, int W, int Q, typename Orb>
__device__ __forceinline__ void ll_hops(const char* lds, PairTab<VT> vk, int L, Orb orb, uint32_t nlo,
                                        const uint32_t* words, const uint32_t* hop, double* acc) {
    constexpr int kWords = doci_ll_words(W);
    uint32_t wd[Q][kWords];
#pragma unroll
    for (int d = 0; d < kWords; ++d)
#pragma unroll
        for (int q = 0; q < Q; ++q) wd[q][d] = (words + (size_t)d * nlo)[hop[q]];
#pragma unroll
    for (int j = 1; j < W; ++j) {
        PairTab<VT> trow = vk + orb(j) * L;
        const int p0 = j * (j - 1) / 2;
#pragma unroll
        for (int k = 0; k < j; ++k) {
            const double v = (double)trow[orb(k)];
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const uint32_t o = wd[q][(p0 + k) / 2];
                acc[q] += v * *(const double*)(lds + ((p0 + k) % 2 ? o >> 16 : o & 0xffffu));
            }
        }
    }
}

// Hops across the split with one stage of either kind; m[q][k]: lanes whose row q
// occupies orbital k.
template <typename VT, int W, int Q, typename Orb>
__device__ __forceinline__ void split_hops(const char* lds, PairTab<VT> ta, PairTab<VT> tb, Orb orb,
                                           const uint32_t (*idx)[(W + 1) / 2], const uint64_t (*m)[W], double* acc) {
#pragma unroll
    for (int k = 0; k < W; ++k) {
        const double va = (double)ta[orb(k)], vb = (double)tb[orb(k)];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const uint32_t off = k % 2 ? idx[q][k / 2] >> 16 : idx[q][k / 2] & 0xffffu;
            acc[q] += (__builtin_amdgcn_inverse_ballot_w64(m[q][k]) ? vb : va) * *(const double*)(lds + off);
        }
    }
}

// High -> high hops: the neighbour block at the same row, several hops' loads in
// flight per row.
template <int Q>
__device__ __forceinline__ void hh_hops(const double* x, const uint32_t* base, const double* val, int nhh,
                                        const uint32_t* roff, double* acc) {
    constexpr int U = Q >= 3 ? 4 : 8;
    for (int t = 0; t < nhh; t += U) {
        double xv[Q][U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const double* xn = x + __builtin_amdgcn_readfirstlane(base[min(t + u, nhh - 1)]);
#pragma unroll
            for (int q = 0; q < Q; ++q) xv[q][u] = at_byte(xn, roff[q]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const double e = t + u < nhh ? val[t + u] : 0.0;
#pragma unroll
            for (int q = 0; q < Q; ++q) acc[q] += e * xv[q][u];
        }
    }
}

template <typename VT, int W, int ROWS, int T, bool BATCH>
__global__ void __launch_bounds__(T) k_spmv_doci_blk(DociBlockArgs a, const VT* __restrict__ vk0,
                                                      const double* __restrict__ x0, double* __restrict__ y0,
                                                      DociBatch bt) {
    constexpr uint32_t kCap = ROWS * T;
    constexpr uint32_t kZero = doci_zero_off(kCap);
    __shared__ __align__(16) char lds[kZero + 8];
    double* xa = (double*)lds;      // the own block, then the high -> low stages
    double* xb = xa + kCap;         // the low -> high stages
    const VT* __restrict__ vk = vk0;
    const double* __restrict__ x = x0;
    double* __restrict__ y = y0;
    const double* __restrict__ diag = a.diag;
    if (BATCH) {  // lane blockIdx.y of a batched Davidson product
        const int lane = blockIdx.y;
        const BdStep& st = bt.step[lane];
        if (st.mode == BD_IDLE || st.f32 != (sizeof(VT) == 4 ? 1 : 0)) return;
        const BdOpLane& o = bt.op[lane];
        vk = sizeof(VT) == 4 ? reinterpret_cast<const VT*>(o.vk32) : reinterpret_cast<const VT*>(o.vk64);
        diag = o.diag;
        const uint64_t off = ((uint64_t)lane * bt.M + st.m) * bt.n;
        x = bt.V + off;
        y = bt.S + off;
    }
    const PairTab<VT> tab = (PairTab<VT>)(uintptr_t)vk;
    const auto* dg = (const __attribute__((address_space(1))) double*)(uintptr_t)diag;
    __shared__ BlockSums sums;
    __shared__ uint32_t hh_base[kBlkHops];
    __shared__ double hh_val[kBlkHops];
    __shared__ uint32_t sg_base[2][kBlkStages], sg_orb[2][kBlkStages];  // high -> low, low -> high
    const int L = a.L, w = a.w, nh = L - w;
    const uint32_t nlo = 1u << w;
    // orbitals w .. W - 1 of an instance for more low orbitals: any pair element, times the zero
    auto orb = [w](int k) { return W <= 7 ? min(k, w - 1) : k; };
    const int tid = threadIdx.x;
    const DociBlock blk = a.blocks[blockIdx.x];
    const uint32_t R = blk.R, base = blk.base, hi = blk.hi;
    const int c = (int)blk.c;
    const uint32_t hv = ~hi & ((1u << nh) - 1);
    const int ch = __builtin_popcount(hi), cv = nh - ch;
    const int nhh = ch * cv;
    // stages: high -> low (block (hi ^ jh, c + 1)) for every occupied high
    // orbital, low -> high (block (hi | kh, c - 1)) for every empty one
    const int n_hl = c < w ? ch : 0, n_lh = c > 0 ? cv : 0, nst = max(n_hl, n_lh);
    const uint32_t R_hl = c < w ? a.lo_off[c + 2] - a.lo_off[c + 1] : 0u;
    const uint32_t R_lh = c > 0 ? a.lo_off[c] - a.lo_off[c - 1] : 0u;
    for (uint32_t t = tid; t < R; t += T) xa[t] = x[base + t];
    if (tid == 0) *(double*)(lds + kZero) = 0.0;
    if (tid < 64) {
        sums.fill(hi, c, w, nh, a.binom);
        sg_base[tid >> 5][tid & 31] = 0;  // stages that are not there
        sg_orb[tid >> 5][tid & 31] = 0;
    }
    // rows of the wavefront: r = tid + q T, q < nq
    const uint32_t wave0 = __builtin_amdgcn_readfirstlane(tid);
    const int nq = R > wave0 ? (int)((R - 1 - wave0) / T) + 1 : 0;
    const uint16_t* lof = a.lo_of + a.lo_off[c];
    uint32_t hop[ROWS], roff[ROWS], idx[ROWS][(W + 1) / 2];
    double acc[ROWS];
    uint64_t m[ROWS][W];
#pragma unroll
    for (int q = 0; q < ROWS; ++q) {
        const uint32_t r = tid + q * T;
        const uint32_t l = r < R ? lof[r] : 0u;
        hop[q] = a.lo_off[c] + min(r, R - 1);
        roff[q] = min(r, R - 1) * 8u;
#pragma unroll
        for (int k = 0; k < W; k += 2)
            idx[q][k / 2] = (a.hops + (size_t)(doci_ll_words(W) + k / 2) * nlo)[hop[q]];
        acc[q] = 0.0;
        if (r < R) {
            double d = dg[base + r];
            if (!(fabs(d) > a.zero)) d = 0.0;
            acc[q] = (double)(VT)d * x[base + r];
        }
#pragma unroll
        for (int k = 0; k < W; ++k) m[q][k] = __ballot((l >> k) & 1u);
    }
    __syncthreads();
    for (int t = tid; t < nh * 32; t += T) {  // neighbour blocks of the hops that leave or stay in the high part
        const int j = t >> 5, k = t & 31;
        if (k >= nh || ((hi >> k) & 1u)) continue;
        const int ik = __builtin_popcount(hv & ((1u << k) - 1));
        if ((hi >> j) & 1u) {
            const int i = __builtin_popcount(hi & ((1u << j) - 1)) * cv + ik;
            hh_base[i] = sums.moved(j, k);
            hh_val[i] = (double)tab[(w + j) * L + (w + k)];
        }
    }
    if (tid < 2 * kBlkStages && (tid & 31) < nh) {
        const int q = tid & 31, dir = tid >> 5;
        const uint32_t set = dir ? hv : hi;
        const int i = __builtin_popcount(set & ((1u << q) - 1));
        if (((set >> q) & 1u) && i < (dir ? n_lh : n_hl)) {
            sg_base[dir][i] = dir ? sums.added(q) : sums.removed(q);
            sg_orb[dir][i] = (uint32_t)(w + q);
        }
    }
    __syncthreads();
    // a pair of stages into registers while the one before is worked on; a stage
    // that is not there is all zeros
    double pa[ROWS], pb[ROWS];
    auto fetch = [&](int s) {
        const uint32_t Ra = s < n_hl ? R_hl : 0u, Rb = s < n_lh ? R_lh : 0u;
        const uint32_t ba = __builtin_amdgcn_readfirstlane(sg_base[0][s]), bb = __builtin_amdgcn_readfirstlane(sg_base[1][s]);
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const uint32_t t = tid + i * T;
            pa[i] = t < Ra ? x[ba + t] : 0.0;
            pb[i] = t < Rb ? x[bb + t] : 0.0;
        }
    };
    if (nst) fetch(0);
    auto rows = [&](auto qc) {
        constexpr int Q = decltype(qc)::value;
        ll_hops<VT, W, Q>(lds, tab, L, orb, nlo, a.hops, hop, acc);
        hh_hops<Q>(x, hh_base, hh_val, nhh, roff, acc);
    };
    auto split = [&](auto qc, int s) {
        PairTab<VT> ta = tab + __builtin_amdgcn_readfirstlane(sg_orb[0][s]) * L;  // symmetric table
        PairTab<VT> tb = tab + __builtin_amdgcn_readfirstlane(sg_orb[1][s]) * L;
        split_hops<VT, W, decltype(qc)::value>(lds, ta, tb, orb, idx, m, acc);
    };
    using std::integral_constant;
    if (ROWS >= 4 && nq >= 3) rows(integral_constant<int, ROWS>());
    else if (ROWS >= 2 && nq >= 2) rows(integral_constant<int, ROWS < 2 ? 1 : 2>());
    else if (nq >= 1) rows(integral_constant<int, 1>());
    for (int s = 0; s < nst; ++s) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            xa[tid + i * T] = pa[i];
            xb[tid + i * T] = pb[i];
        }
        __syncthreads();
        if (s + 1 < nst) fetch(s + 1);
        if (ROWS >= 4 && nq >= 3) split(integral_constant<int, ROWS>(), s);
        else if (ROWS >= 2 && nq >= 2) split(integral_constant<int, ROWS < 2 ? 1 : 2>(), s);
        else if (nq >= 1) split(integral_constant<int, 1>(), s);
    }
#pragma unroll
    for (int q = 0; q < ROWS; ++q) {
        const uint32_t r = tid + q * T;
        if (r < R) y[base + r] = acc[q];
    }
}

// The same product walking the set bits of each row's low pattern: work in
// proportion to the hops a row has, 62 VGPRs, many workgroups a CU.  Away from
// half filling most blocks are small and few orbital pairs of a row are hops (see
// doci_walks).
constexpr int kBlkRows = 1024;  // LDS x block capacity (>= C(12, 6))

__device__ __forceinline__ uint32_t doci_block_base(uint32_t hi, int c, int w, const uint64_t* __restrict__ binom) {
    uint32_t b = 0;
    int m = c + 1;
    for (uint32_t t = hi; t; t &= t - 1) {
        b += (uint32_t)binom[(w + __builtin_ctz(t)) * kBinomCols + m];
        ++m;
    }
    return b;
}

__device__ __forceinline__ int nth_bit(uint32_t v, int k) {  // position of the k-th (0-based) set bit
    for (int i = 0; i < k; ++i) v &= v - 1;
    return __builtin_ctz(v);
}

template <typename VT, int ROWS, int T, bool BATCH>
__global__ void __launch_bounds__(T) k_spmv_doci_walk(DociBlockArgs a, const VT* __restrict__ vk0,
                                                      const double* __restrict__ x0, double* __restrict__ y0,
                                                      DociBatch bt) {
    extern __shared__ double smem_blk[];
    const VT* __restrict__ vk = vk0;
    const double* __restrict__ x = x0;
    double* __restrict__ y = y0;
    const double* __restrict__ diag = a.diag;
    if (BATCH) {  // lane blockIdx.y of a batched Davidson product
        const int lane = blockIdx.y;
        const BdStep& st = bt.step[lane];
        if (st.mode == BD_IDLE || st.f32 != (sizeof(VT) == 4 ? 1 : 0)) return;
        const BdOpLane& o = bt.op[lane];
        vk = sizeof(VT) == 4 ? reinterpret_cast<const VT*>(o.vk32) : reinterpret_cast<const VT*>(o.vk64);
        diag = o.diag;
        const uint64_t off = ((uint64_t)lane * bt.M + st.m) * bt.n;
        x = bt.V + off;
        y = bt.S + off;
    }
    __shared__ uint32_t hh_base[kBlkHops];
    __shared__ double hh_val[kBlkHops];
    __shared__ uint32_t sg_base[kBlkStages], sg_orb[kBlkStages];
    const int L = a.L, w = a.w, nh = L - w;
    const uint32_t W = 1u << w, wmask = W - 1;
    // one x buffer: the own block, then each staged block in turn; a barrier
    // before every stage's write lets all threads finish reading the previous
    // contents (one buffer instead of three leaves room for more resident
    // workgroups per CU, the kernel's limit)
    double* xo = smem_blk;
    double* sbuf = smem_blk;
    VT* tab = reinterpret_cast<VT*>(smem_blk + kBlkRows);
    uint16_t* rlo = reinterpret_cast<uint16_t*>(tab + L * L);
    const int tid = threadIdx.x;
    const DociBlock blk = a.blocks[blockIdx.x];
    const uint32_t R = blk.R, base = blk.base, hi = blk.hi;
    const int c = (int)blk.c;
    const uint32_t hv = ~hi & ((1u << nh) - 1);
    const int ch = __builtin_popcount(hi), cv = nh - ch;
    const int nhh = ch * cv;
    // stages: high -> low (block (hi ^ jh, c + 1)) for every occupied high
    // orbital, then low -> high (block (hi | kh, c - 1)) for every empty one
    const int n_hl = c < w ? ch : 0, n_lh = c > 0 ? cv : 0, nst = n_hl + n_lh;
    const uint32_t R_hl = c < w ? a.lo_off[c + 2] - a.lo_off[c + 1] : 0u;
    const uint32_t R_lh = c > 0 ? a.lo_off[c] - a.lo_off[c - 1] : 0u;
    for (int t = tid; t < L * L; t += T) tab[t] = vk[t];
    for (uint32_t t = tid; t < W; t += T) rlo[t] = a.rank_lo[t];
    for (uint32_t t = tid; t < R; t += T) xo[t] = x[base + t];
    if (tid < nhh) {  // neighbour blocks of the high -> high hops, one per thread
        const int jh = nth_bit(hi, tid / cv), kh = nth_bit(hv, tid % cv);
        hh_base[tid] = doci_block_base(hi ^ (1u << jh) ^ (1u << kh), c, w, a.binom);
        hh_val[tid] = (double)vk[(w + jh) * L + (w + kh)];
    }
    if (tid < nst) {
        if (tid < n_hl) {
            const int jh = nth_bit(hi, tid);
            sg_base[tid] = doci_block_base(hi ^ (1u << jh), c + 1, w, a.binom);
            sg_orb[tid] = (uint32_t)(w + jh);
        } else {
            const int kh = nth_bit(hv, tid - n_hl);
            sg_base[tid] = doci_block_base(hi | (1u << kh), c - 1, w, a.binom);
            sg_orb[tid] = (uint32_t)(w + kh);
        }
    }
    const uint16_t* lof = a.lo_of + a.lo_off[c];
    uint32_t lo[ROWS];
    double acc[ROWS];
#pragma unroll
    for (int q = 0; q < ROWS; ++q) {
        const uint32_t r = tid + q * T;
        lo[q] = r < R ? lof[r] : 0u;
        acc[q] = 0.0;
    }
    __syncthreads();
    // first staged block into registers while the own block is worked on
    double pre[ROWS];
    auto fetch = [&](int sidx) {
        const uint32_t Rs = sidx < n_hl ? R_hl : R_lh, b = sg_base[sidx];
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const uint32_t t = tid + i * T;
            pre[i] = t < Rs ? x[b + t] : 0.0;
        }
    };
    if (nst) fetch(0);
    // diagonal and low -> low hops
#pragma unroll
    for (int q = 0; q < ROWS; ++q) {
        const uint32_t r = tid + q * T;
        if (r < R) {
            double d = diag[base + r];
            if (!(fabs(d) > a.zero)) d = 0.0;
            double s = (double)(VT)d * xo[r];
            const uint32_t l = lo[q], vl = ~l & wmask;
            for (uint32_t o = l; o; o &= o - 1) {
                const int j = __builtin_ctz(o);
                const uint32_t lj = l ^ (1u << j);
                const VT* trow = tab + j * L;
                for (uint32_t v = vl; v; v &= v - 1) {
                    const int k = __builtin_ctz(v);
                    s += (double)trow[k] * xo[rlo[lj | (1u << k)]];
                }
            }
            acc[q] = s;
        }
    }
    // high -> high hops: the neighbour block at the same row index, four
    // hops' loads in flight per row
    {
        int t = 0;
        for (; t + 4 <= nhh; t += 4) {
            const uint32_t b0 = hh_base[t], b1 = hh_base[t + 1], b2 = hh_base[t + 2], b3 = hh_base[t + 3];
            const double e0 = hh_val[t], e1 = hh_val[t + 1], e2 = hh_val[t + 2], e3 = hh_val[t + 3];
#pragma unroll
            for (int q = 0; q < ROWS; ++q) {
                const uint32_t r = tid + q * T;
                if (r < R) {
                    const double x0 = x[b0 + r], x1 = x[b1 + r], x2 = x[b2 + r], x3 = x[b3 + r];
                    acc[q] += e0 * x0 + e1 * x1 + e2 * x2 + e3 * x3;
                }
            }
        }
        for (; t < nhh; ++t) {
            const uint32_t b0 = hh_base[t];
            const double e0 = hh_val[t];
#pragma unroll
            for (int q = 0; q < ROWS; ++q) {
                const uint32_t r = tid + q * T;
                if (r < R) acc[q] += e0 * x[b0 + r];
            }
        }
    }
    // staged hops across the split: stage s+1 loads into registers while
    // stage s is read from LDS; two barriers per stage
    for (int sidx = 0; sidx < nst; ++sidx) {
        double* buf = sbuf;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ROWS; ++i) buf[tid + i * T] = pre[i];
        __syncthreads();
        if (sidx + 1 < nst) fetch(sidx + 1);
        const int orb = (int)sg_orb[sidx];
        const VT* trow = tab + orb * L;  // pair elements with the high orbital (symmetric table)
        if (sidx < n_hl) {  // high orbital orb -> empty low orbital k
#pragma unroll
            for (int q = 0; q < ROWS; ++q) {
                const uint32_t r = tid + q * T;
                if (r < R) {
                    const uint32_t l = lo[q];
                    double s = 0.0;
                    for (uint32_t v = ~l & wmask; v; v &= v - 1) {
                        const int k = __builtin_ctz(v);
                        s += (double)trow[k] * buf[rlo[l | (1u << k)]];
                    }
                    acc[q] += s;
                }
            }
        } else {  // occupied low orbital j -> empty high orbital orb
#pragma unroll
            for (int q = 0; q < ROWS; ++q) {
                const uint32_t r = tid + q * T;
                if (r < R) {
                    const uint32_t l = lo[q];
                    double s = 0.0;
                    for (uint32_t o = l; o; o &= o - 1) {
                        const int j = __builtin_ctz(o);
                        s += (double)trow[j] * buf[rlo[l ^ (1u << j)]];
                    }
                    acc[q] += s;
                }
            }
        }
    }
#pragma unroll
    for (int q = 0; q < ROWS; ++q) {
        const uint32_t r = tid + q * T;
        if (r < R) y[base + r] = acc[q];
    }
}

// Fillings on the bit-walking kernel: below a third (or above two thirds), with
// twelve low orbitals below 5/12.  Walking / tabled, FP64, us, w < 12: L=22 6 pairs
// 24.7 / 23.9, L=23 7 pairs 45 / 46, L=21 7 pairs 19.9 / 18.5, L=23 8 pairs 60 / 59,
// L=22 8 pairs 38 / 34, L=20 8 pairs 17.0 / 12.9, L=23 11 pairs 95 / 81; w = 12:
// L=31 5 pairs 218 / 459, L=24 8 pairs 100 / 117, L=26 10 pairs 568 / 598, L=27 11
// pairs 1369 / 1388, L=26 11 pairs 705 / 683, L=24 12 pairs 195 / 174.
static bool doci_walks(int L, int np, int w) {
    const int m = np < L - np ? np : L - np;
    return w == 12 ? 12 * m < 5 * L : 3 * m < L;
}

int doci_block_w(int L) { return L / 2 < kDociMaxW ? L / 2 : kDociMaxW; }

template <typename VT, bool BATCH>
static void launch_doci_blk_t(const DociBlockArgs& a, const VT* vk, const double* x, double* y, hipStream_t s,
                              const DociBatch& bt, int lanes) {
    if (!a.nblocks) return;
    CF_REQUIRE(a.w >= 1 && a.w <= kDociMaxW && a.L - a.w >= 1 && a.L - a.w <= 20,
               "block-staged DOCI SpMV: 1 <= w <= 12 low orbitals and 1..20 high orbitals");
    const dim3 g(a.nblocks, (unsigned)lanes);
    if (doci_walks(a.L, a.np, a.w)) {
        const size_t shm = kBlkRows * sizeof(double) + (size_t)a.L * a.L * sizeof(VT) +
                           ((size_t)1 << a.w) * sizeof(uint16_t);
        // rows of the largest block over the workgroup (T * ROWS >= C(w, w/2)); the
        // neighbour-block bases are computed one per thread (T >= ch (nh - ch))
        const uint64_t maxR = binom_host(a.w, a.w / 2);
        const int nh = a.L - a.w, maxhh = (nh / 2) * ((nh + 1) / 2);
        if (maxR <= 64 && maxhh <= 64) k_spmv_doci_walk<VT, 1, 64, BATCH><<<g, 64, shm, s>>>(a, vk, x, y, bt);
        else if (maxR <= 128 && maxhh <= 128) k_spmv_doci_walk<VT, 1, 128, BATCH><<<g, 128, shm, s>>>(a, vk, x, y, bt);
        else if (maxR <= 256) k_spmv_doci_walk<VT, 1, 256, BATCH><<<g, 256, shm, s>>>(a, vk, x, y, bt);
        else if (maxR <= 512) k_spmv_doci_walk<VT, 2, 256, BATCH><<<g, 256, shm, s>>>(a, vk, x, y, bt);
        else k_spmv_doci_walk<VT, 4, 256, BATCH><<<g, 256, shm, s>>>(a, vk, x, y, bt);
        CF_HIP(hipGetLastError());
        return;
    }
    // rows of the largest block over the workgroup: T * ROWS >= C(w, w/2)
    if (a.w <= 7) k_spmv_doci_blk<VT, 7, 1, 64, BATCH><<<g, 64, 0, s>>>(a, vk, x, y, bt);
    else if (a.w <= 9) k_spmv_doci_blk<VT, 9, 1, 128, BATCH><<<g, 128, 0, s>>>(a, vk, x, y, bt);
    else if (a.w <= 10) k_spmv_doci_blk<VT, 10, 1, 256, BATCH><<<g, 256, 0, s>>>(a, vk, x, y, bt);
    else if (a.w <= 11) k_spmv_doci_blk<VT, 11, 2, 256, BATCH><<<g, 256, 0, s>>>(a, vk, x, y, bt);
    else k_spmv_doci_blk<VT, 12, 2, 512, BATCH><<<g, 512, 0, s>>>(a, vk, x, y, bt);
    CF_HIP(hipGetLastError());
}

template <typename VT>
static void launch_doci_blk(const DociBlockArgs& a, const VT* vk, const double* x, double* y, hipStream_t s) {
    launch_doci_blk_t<VT, false>(a, vk, x, y, s, DociBatch{}, 1);
}

void launch_spmv_doci_blk_batch(const DociBlockArgs& a, bool f32, const DociBatch& bt, int lanes, hipStream_t s) {
    CF_REQUIRE(lanes >= 1 && lanes <= kBdMaxLanes, "batched DOCI product: 1..32 lanes");
    if (f32) launch_doci_blk_t<float, true>(a, nullptr, nullptr, nullptr, s, bt, lanes);
    else launch_doci_blk_t<double, true>(a, nullptr, nullptr, nullptr, s, bt, lanes);
}

void launch_spmv_doci_blk_f64(const DociBlockArgs& a, const double* vk, const double* x, double* y, hipStream_t s) {
    launch_doci_blk<double>(a, vk, x, y, s);
}

void launch_spmv_doci_blk_f32(const DociBlockArgs& a, const float* vk, const double* x, double* y, hipStream_t s) {
    launch_doci_blk<float>(a, vk, x, y, s);
}

void launch_spmv_doci_f64(const DociEllArgs& a, DociShape sh, const double* vk, const double* x, double* y,
                          hipStream_t s) {
    launch_doci<double>(a, sh, vk, x, y, s);
}

void launch_spmv_doci_f32(const DociEllArgs& a, DociShape sh, const float* vk, const double* x, double* y,
                          hipStream_t s) {
    launch_doci<float>(a, sh, vk, x, y, s);
}

}  // namespace cf
