// The alpha-beta part of the FCI sigma as a matrix product (FP64 operands).
//
//   sigma_ab(Ia, Ib) = sum_{a in A(Ia)} sum_{b in A(Ib)} s_a s_b V[p_a][q_b][r_a][s_b] C(J_a, J_b)
//
// (see sigma.hip).  For a fixed Ia the alpha actions are fixed, and V is
// symmetric in q <-> s for real orbitals, so with the unordered pairs {q, s}
//   F(J, {qs}) = sum_{a in A(Ia)} C(J_a, J) s_a V[p_a][q][r_a][s]
// is a d_b x |A| by |A| x L(L+1)/2 product on FP64 MFMA -- the number operators
// of Ia are one action with the slice summed over its electrons -- and
//   sigma_ab(Ia, Ib) = sum_{b in A(Ib)} s_b F(J_b, {q_b s_b})
// takes one LDS read per beta action.  Applying the actions pair by pair took
// two LDS reads per term: |A| times as many, which is what bounded it.
//
// A workgroup of eight wavefronts owns one Ia.  The rows C(J_a, .) are read
// once, straight into the MFMA operand registers (16 consecutive elements of
// four rows per load), the |A| x pairs matrix goes to LDS, and F is made 16
// columns at a time: MFMAs, F to LDS, the gathers of the beta actions that lie
// in those columns (sorted by column once per space).  Up to two pairs left
// over a multiple of 16 are summed on the VALU instead of in a tile of their own
// (L=11: 66 = 4 * 16 + 2).
//
// Bound by the MFMAs: 2 * 16 ceil(d_b / 16) * 4 ceil(|A| / 4) * 16 tiles flop per Ia.
// L=12 (6,6), d = 853,776: 188 us, whole sigma 243 us (433 with ab3's pair by
// pair actions); 12 vectors of L=11 (5,5), d = 213,444: 353 us (627).  The
// MFMAs alone are 79 and 151 us at the card's 69.4 TFLOP/s, the rest the gathers
// and the barriers around them.  Two of the instances are at the limit of their
// registers: <8, 4> (L=11) spills 4 of 128 VGPRs, <10, 8> (L=12) 8 of 256.
#include "sigma.h"

#include <algorithm>

namespace cf {

namespace {

typedef double v4ds __attribute__((ext_vector_type(4)));
constexpr int kWaves = 8, kThreads = kWaves * 64;
constexpr int kFS = 17;  // row stride of F in LDS
constexpr int kMaxTiles = 16;  // L <= 16: 136 pairs, 9 tiles
static_assert(kSigmaStarts >= 2 * kMaxTiles + 1, "starts and longest lists");

__device__ __forceinline__ int pair_col(int a, int b) {
    const int q = a > b ? a : b, s = a > b ? b : a;
    return q * (q + 1) / 2 + s;
}

struct MfmaShape {
    int np = 0;      // pairs
    int tiles = 0;   // tiles of 16 columns on MFMA
    int rem = 0;     // columns summed on the VALU after them
    int bs = 0;      // LDS row stride of the |A| x pairs matrix
    int ks = 0;      // k-steps of 4 actions
    int rows = 0;    // d_b rounded up to 16
    size_t lds = 0;
};

MfmaShape shape_of(const SigmaArgs& a) {
    MfmaShape m;
    m.np = a.L * (a.L + 1) / 2;
    m.rem = m.np % 16 <= 2 ? m.np % 16 : 0;
    m.tiles = m.rem ? m.np / 16 : (m.np + 15) / 16;
    m.bs = m.tiles * 16 + m.rem;
    if (2 * m.bs % 64 < 12) m.bs += m.rem ? 4 : 8;  // the four rows of a read on different banks
    m.ks = std::max(4, (a.Sa + 3) / 4);  // the smallest instance has four
    m.rows = (int)((a.db + 15) / 16 * 16);
    m.lds = ((size_t)(m.rows + 1) * kFS + (size_t)m.ks * 4 * m.bs) * sizeof(double);
    return m;
}

// Beta actions of each string sorted by column tile: gat[slot][db] = byte
// offset of F(J, column in tile) | sign << 31.  A tile's slots are the same for
// every string -- gst[tile] .. gst[tile + 1], as many as the longest list, in
// fours, the rest pointing at a row of zeros -- so that several codes and LDS
// reads are in flight at once.  k_mfma_count finds the longest lists (at most
// 16: a string has one action per pair), k_mfma_gather fills.  (Codes of 16
// bits, all of a tile's loaded before the barrier, spilled more: 204 us instead of
// 183 at L=12, and no gain at L=11.)
template <class Put>
__device__ __forceinline__ void beta_actions(const Exc* l, int Sb, uint32_t Ib, str_t bits, Put&& put) {
    for (int e = 0; e < Sb; ++e)
        if (l[e].type == 1) put(l[e].J, pair_col(l[e].f, l[e].t), l[e].sign < 0);
    for (str_t u = bits; u; u &= u - 1) put(Ib, pair_col(__builtin_ctzll(u), __builtin_ctzll(u)), false);
}

__global__ void __launch_bounds__(256) k_mfma_count(uint64_t db, int Sb, const str_t* __restrict__ sb,
                                                    const Exc* __restrict__ subb, uint32_t* __restrict__ most) {
    const uint64_t Ib = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    const int t = blockIdx.y;
    uint32_t n = 0;
    if (Ib < db)
        beta_actions(subb + Ib * (uint64_t)Sb, Sb, (uint32_t)Ib, sb[Ib],
                     [&](uint32_t, int col, bool) { n += col / 16 == t ? 1 : 0; });
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) n = max(n, __shfl_xor(n, o, 64));
    if ((threadIdx.x & 63) == 0) atomicMax(&most[t], n);
}

__global__ void __launch_bounds__(256) k_mfma_gather(uint64_t db, int Sb, int rows, const str_t* __restrict__ sb,
                                                     const Exc* __restrict__ subb, const uint32_t* __restrict__ most,
                                                     uint32_t* __restrict__ gst, uint32_t* __restrict__ gat) {
    const uint64_t Ib = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    const int t = blockIdx.y;
    uint32_t n = 0;
    for (int c = 0; c < t; ++c) n += (most[c] + 3) / 4 * 4;
    const uint32_t end = n + (most[t] + 3) / 4 * 4;
    if (Ib == 0) {
        gst[t] = n;
        if (blockIdx.y + 1 == gridDim.y) gst[t + 1] = end;
    }
    if (Ib >= db) return;
    beta_actions(subb + Ib * (uint64_t)Sb, Sb, (uint32_t)Ib, sb[Ib], [&](uint32_t J, int c, bool neg) {
        if (c / 16 != t) return;
        gat[(uint64_t)n++ * db + Ib] = (J * kFS + (uint32_t)(c % 16)) * 8u | (neg ? 0x80000000u : 0u);
    });
    for (; n < end; ++n) gat[(uint64_t)n * db + Ib] = (uint32_t)(rows * kFS) * 8u;  // the row of zeros
}

// *sym = 1 if V[p][q][r][s] = V[p][s][r][q] to rounding: 2^-50 of the largest
// element.  Integrals over real orbitals, whose rotations differ by 5.1e-16 of it
// at most (L = 4 .. 16, six sets, small and large rotations).  The product takes
// the mean of the two, so what it takes differs from what it was given by half
// of that: 1e-16 relative in the result of rotated integrals, below its sums'
// rounding.
__global__ void __launch_bounds__(1024) k_v_symmetric(int L, const double* __restrict__ V, int* sym) {
    __shared__ double red[16];
    __shared__ int bad;
    const int L2 = L * L, L4 = L2 * L2;
    double m = 0.0;
    for (int i = threadIdx.x; i < L4; i += 1024) m = fmax(m, fabs(V[i]));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    if (threadIdx.x == 0) bad = 0;
    __syncthreads();
    for (int i = 0; i < 16; ++i) m = fmax(m, red[i]);
    const double most = 0x1p-50 * m;
    for (int i = threadIdx.x; i < L4; i += 1024) {
        const int p = i / (L2 * L), q = i / L2 % L, r = i / L % L, s = i % L;
        if (q > s && !(fabs(V[i] - V[((p * L + s) * L + r) * L + q]) <= most)) bad = 1;
    }
    __syncthreads();
    if (threadIdx.x == 0) *sym = bad ? 0 : 1;
}

template <int KS, int RT, bool BATCH>
__global__ void __launch_bounds__(kThreads, RT <= 4 && KS <= 8 ? 4 : 2)
    k_sigma_mfma(SigmaArgs a0, const double* __restrict__ C0, double* __restrict__ sig0, SigmaBatch sb, MfmaShape m) {
    extern __shared__ double smem_ab4[];
    SigmaArgs a = a0;
    const double* __restrict__ C = C0;
    double* __restrict__ sig = sig0;
    if (BATCH) {
        const int lane = blockIdx.y;
        const BdStep& st = sb.step[lane];
        if (st.mode == BD_IDLE || st.f32) return;
        a = sb.args[lane];
        if (!a.sym) return;
        const uint64_t off = ((uint64_t)lane * sb.M + st.m) * sb.n;
        C = sb.V + off;
        sig = sb.S + off;
    }
    const uint32_t per = gridDim.x >> 3;
    const uint32_t Ia = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if (Ia >= a.da) return;
    const int db = (int)a.db, L = a.L, L2 = L * L, Sa = a.Sa;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int r = lane & 15, kq = lane >> 4;
    double* F = smem_ab4;
    double* B = F + (m.rows + 1) * kFS;
    const Exc* la = a.suba + (uint64_t)Ia * Sa;
    // operand rows: element [t][k] = C(J_a, 16 (w + 8 t) + r), a = 4 k + kq
    double av[RT][KS];
    {
        const double* row[KS];
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const int e = 4 * k + kq;
            row[k] = C + (uint64_t)(e < Sa ? la[e].J : Ia) * db;
        }
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            const int j = 16 * (w + kWaves * t) + r;
#pragma unroll
            for (int k = 0; k < KS; ++k) av[t][k] = j < db ? row[k][j] : 0.0;
        }
    }
    // B[a][{qs}] = s_a V[p_a][q][r_a][s] (the mean of the two orders), zeros past the actions and pairs
    for (int e = w; e < KS * 4; e += kWaves) {
        const Exc x = la[e < Sa ? e : 0];
        const double* v = x.type == 0 ? a.vself64 + (uint64_t)Ia * L2 : a.vpair64 + (uint64_t)(x.f * L + x.t) * L2;
        const bool neg = x.type == 1 && x.sign < 0;
        for (int c = lane; c < m.bs; c += 64) {
            double y = 0.0;
            if (e < Sa && c < m.np) {
                const int q = (int)((sqrtf(8 * c + 1.5f) - 1.0f) * 0.5f);  // c >= q (q + 1) / 2
                const int s = c - q * (q + 1) / 2;
                y = 0.5 * (v[q * L + s] + v[s * L + q]);
            }
            B[e * m.bs + c] = neg ? -y : y;
        }
    }
    if (tid < kFS) F[m.rows * kFS + tid] = 0.0;
    __syncthreads();
    constexpr int IB = (RT * 16 * kWaves + kThreads - 1) / kThreads;  // beta strings a thread gathers for
    double acc[IB];
#pragma unroll
    for (int i = 0; i < IB; ++i) acc[i] = 0.0;
    const int ntile = m.tiles + (m.rem ? 1 : 0);
    for (int ct = 0; ct < ntile; ++ct) {
        if (ct < m.tiles) {
            v4ds f[RT];
#pragma unroll
            for (int t = 0; t < RT; ++t) f[t] = v4ds{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int k = 0; k < KS; ++k) {
                const double bv = B[(4 * k + kq) * m.bs + ct * 16 + r];
#pragma unroll
                for (int t = 0; t < RT; ++t)
                    f[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[t][k], bv, f[t], 0, 0, 0);
            }
            __syncthreads();  // the last columns have been gathered
#pragma unroll
            for (int t = 0; t < RT; ++t) {
                const int j0 = 16 * (w + kWaves * t);
                if (j0 < m.rows) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) F[(j0 + 4 * v + kq) * kFS + r] = f[t][v];
                }
            }
        } else {  // the one or two pairs left over: sums over the lanes' actions
            __syncthreads();
            for (int c = 0; c < m.rem; ++c) {
#pragma unroll
                for (int t = 0; t < RT; ++t) {
                    double s = 0.0;
#pragma unroll
                    for (int k = 0; k < KS; ++k) s = fma(av[t][k], B[(4 * k + kq) * m.bs + ct * 16 + c], s);
                    s += __shfl_xor(s, 16, 64);
                    s += __shfl_xor(s, 32, 64);
                    const int j0 = 16 * (w + kWaves * t);
                    if (kq == 0 && j0 < m.rows) F[(j0 + r) * kFS + c] = s;
                }
            }
        }
        __syncthreads();
        const uint32_t s1 = a.gst[ct + 1];
        for (uint32_t s = a.gst[ct]; s < s1; s += 4) {
            uint32_t c[IB][4];
#pragma unroll
            for (int i = 0; i < IB; ++i)
#pragma unroll
                for (int u = 0; u < 4; ++u) c[i][u] = a.gat[(uint64_t)(s + u) * db + min(tid + i * kThreads, db - 1)];
#pragma unroll
            for (int i = 0; i < IB; ++i)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const double v = *(const double*)((const unsigned char*)F + (c[i][u] & 0x7fffffffu));
                    acc[i] += __hiloint2double(__double2hiint(v) ^ (int)(c[i][u] & 0x80000000u), __double2loint(v));
                }
        }
    }
#pragma unroll
    for (int i = 0; i < IB; ++i) {
        const int Ib = tid + i * kThreads;
        if (Ib < db) sig[(uint64_t)Ia * db + Ib] += acc[i];
    }
}

template <int KS, int RT>
void launch_t(const SigmaArgs& a, const MfmaShape& m, const double* C, double* sig, const SigmaBatch* sb, int lanes,
              hipStream_t s) {
    const unsigned grid = (unsigned)((a.da + 7) / 8 * 8);
    const void* f = sb ? (const void*)k_sigma_mfma<KS, RT, true> : (const void*)k_sigma_mfma<KS, RT, false>;
    if (m.lds > 64 * 1024) CF_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)m.lds));
    if (sb) k_sigma_mfma<KS, RT, true><<<dim3(grid, (unsigned)lanes), kThreads, m.lds, s>>>(a, nullptr, nullptr, *sb, m);
    else k_sigma_mfma<KS, RT, false><<<grid, kThreads, m.lds, s>>>(a, C, sig, SigmaBatch{}, m);
    CF_HIP(hipGetLastError());
}

template <int KS>
void launch_k(const SigmaArgs& a, const MfmaShape& m, const double* C, double* sig, const SigmaBatch* sb, int lanes,
              hipStream_t s) {
    const int rt = (m.rows / 16 + kWaves - 1) / kWaves;
    if (rt <= 1) launch_t<KS, 1>(a, m, C, sig, sb, lanes, s);
    else if (rt <= 2) launch_t<KS, 2>(a, m, C, sig, sb, lanes, s);
    else if (rt <= 4) launch_t<KS, 4>(a, m, C, sig, sb, lanes, s);
    else launch_t<KS, 8>(a, m, C, sig, sb, lanes, s);
}

}  // namespace

bool sigma_mfma_fits(const SigmaArgs& a) {
    if (a.L > 16 || a.db > 1024 || a.Sa > 40 || !a.da || !a.db || a.da > 0x7ffffff0ull) return false;
    return shape_of(a).lds <= 160 * 1024;
}

uint64_t sigma_mfma_slots(const SigmaArgs& a) {
    const MfmaShape m = shape_of(a);
    return (uint64_t)(m.tiles + (m.rem ? 1 : 0)) * 16 * a.db;
}

void launch_mfma_gather(const SigmaArgs& a, uint32_t* gat, uint32_t* gst, hipStream_t s) {
    const MfmaShape m = shape_of(a);
    const int nt = m.tiles + (m.rem ? 1 : 0);
    if (nt > kMaxTiles) throw Error(ERR_UNSUPPORTED, "sigma: too many pair columns");
    const dim3 g((unsigned)((a.db + 255) / 256), (unsigned)nt);
    uint32_t* most = gst + kMaxTiles + 1;  // longest lists, past the starts
    CF_HIP(hipMemsetAsync(most, 0, kMaxTiles * sizeof(uint32_t), s));
    k_mfma_count<<<g, 256, 0, s>>>(a.db, a.Sb, a.sb, a.subb, most);
    CF_HIP(hipGetLastError());
    k_mfma_gather<<<g, 256, 0, s>>>(a.db, a.Sb, m.rows, a.sb, a.subb, most, gst, gat);
    CF_HIP(hipGetLastError());
}

void launch_v_symmetric(int L, const double* V, int* sym, hipStream_t s) {
    if (L > 64) throw Error(ERR_UNSUPPORTED, "V symmetry test: L <= 64");
    k_v_symmetric<<<1, 1024, 0, s>>>(L, V, sym);
    CF_HIP(hipGetLastError());
}

static void launch_any(const SigmaArgs& a, const double* C, double* sig, const SigmaBatch* sb, int lanes,
                       hipStream_t s) {
    if (!sigma_mfma_fits(a)) throw Error(ERR_UNSUPPORTED, "sigma: shape without a matrix-product kernel");
    const MfmaShape m = shape_of(a);
    if (m.ks == 4) launch_k<4>(a, m, C, sig, sb, lanes, s);
    else if (m.ks == 5) launch_k<5>(a, m, C, sig, sb, lanes, s);
    else if (m.ks == 6) launch_k<6>(a, m, C, sig, sb, lanes, s);
    else if (m.ks == 7) launch_k<7>(a, m, C, sig, sb, lanes, s);
    else if (m.ks == 8) launch_k<8>(a, m, C, sig, sb, lanes, s);
    else if (m.ks == 9) launch_k<9>(a, m, C, sig, sb, lanes, s);
    else launch_k<10>(a, m, C, sig, sb, lanes, s);
}

void launch_sigma_mfma(const SigmaArgs& a, const double* C, double* sig, hipStream_t s) {
    launch_any(a, C, sig, nullptr, 1, s);
}

void launch_sigma_mfma_batch(const SigmaArgs& shape, const SigmaBatch& sb, int lanes, hipStream_t s) {
    if (lanes < 1 || lanes > kBdMaxLanes) throw Error(ERR_ARG, "batched sigma: 1..32 lanes");
    launch_any(shape, nullptr, nullptr, &sb, lanes, s);
}

}  // namespace cf
