// Rows of a determinant list (selected CI) from tables of its strings.
//
// A row's columns are the list determinants at most two excitations away
// (get_ham_element, CIMethod.cpp:459-487).  Looking each of them up in the
// sorted keys costs a binary search -- a chain of a dozen dependent loads -- per
// candidate, twice (count and fill), with the element evaluated from the bit
// strings and the row sorted afterwards.  Here the list's distinct alpha and
// beta strings get their connections among themselves once (popcounts of all
// pairs: some thousand strings at most), with the phases and the one-string
// parts of the elements, and pos[alpha][beta] holds the list index of each
// determinant.  A row then runs over the alpha connections of its alpha string
// and, for each, over the beta connections that keep it within two excitations
// -- itself: all, single: itself and singles, double: itself -- with one load of
// pos per candidate, in ascending (up, down) order, so a sorted list's rows need
// no sort.
//
// Element formulas and orientations are those of k_det_rows (the smaller list
// index first), so the CRS is the same bit for bit.
//
// What bounds it: two dependent loads from L2 (connection, pos) per candidate
// and one for the element.  95,040 determinants of L=12 6a5b (120 alpha strings
// times every beta string; all of the 9.2e7 candidates are stored): 4.7 ms per pass by
// lookup and 2.6 ms for the sort, now 0.78 (count) + 0.92 ms (fill); build, sliced
// copy and first product 15.0 -> 3.25 ms.  Random lists: 95,000 of L=13 6.9 ->
// 4.7 ms, 30,000 of L=10 4.1 -> 1.6 ms.  The tables' launches cost 0.1 ms, which
// lists of 2,000 determinants with many strings do not get back (0.50 -> 0.58 ms
// at 1 in 32 of the pairs), so those stay on the lookup.
#include "dets.h"

#include <algorithm>

#include <hipcub/hipcub.hpp>

#include "string_ops.h"

namespace cf {

namespace {

// first[t] = 1 where sorted entry t begins another value of key >> shift;
// dup counts entries equal to their predecessor.
__global__ void __launch_bounds__(256) k_first(uint64_t n, const uint64_t* __restrict__ key, int shift,
                                               uint32_t* __restrict__ first, unsigned int* dup) {
    const uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    const bool in = t < n;
    const uint64_t k = in ? key[t] : 0, p = in && t > 0 ? key[t - 1] : ~k;
    if (in) first[t] = (k >> shift) != (p >> shift) ? 1u : 0u;
    const uint64_t m = __ballot(in && t > 0 && k == p);
    if (dup && m && (threadIdx.x & 63) == 0) atomicAdd(dup, (unsigned int)__popcll(m));
}

__global__ void __launch_bounds__(256) k_strings_of(uint64_t n, const uint64_t* __restrict__ key, int shift,
                                                    const uint32_t* __restrict__ first,
                                                    const int64_t* __restrict__ at, uint64_t* __restrict__ s) {
    const uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (t < n && first[t]) s[at[t]] = key[t] >> shift;
}

__device__ __forceinline__ uint32_t index_of(const uint64_t* __restrict__ s, uint64_t n, uint64_t v) {
    uint64_t lo = 0, hi = n;
    while (hi - lo > 1) {
        const uint64_t mid = (lo + hi) >> 1;
        if (s[mid] <= v) lo = mid;
        else hi = mid;
    }
    return (uint32_t)lo;
}

__global__ void __launch_bounds__(256) k_det_index(uint64_t n, const str_t* __restrict__ up,
                                                   const str_t* __restrict__ down, const uint64_t* __restrict__ sa,
                                                   uint64_t na, const uint64_t* __restrict__ sb, uint64_t nb,
                                                   uint32_t* __restrict__ ia, uint32_t* __restrict__ ib,
                                                   uint32_t* __restrict__ pos) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const uint32_t a = index_of(sa, na, up[i]), b = index_of(sb, nb, down[i]);
    ia[i] = a;
    ib[i] = b;
    pos[(uint64_t)a * nb + b] = (uint32_t)i;
}

__global__ void __launch_bounds__(256) k_fill_u32(uint64_t n, uint32_t v, uint32_t* __restrict__ out) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = v;
}

__global__ void __launch_bounds__(256) k_narrow_down(uint64_t n, const uint64_t* __restrict__ key,
                                                     uint64_t* __restrict__ out) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = key[i] & 0xffffffffull;
}

// Same-spin double element, two_diff_orbitals(s1, s2) (CIMethod.cpp:429-442).
__device__ __forceinline__ double two_same(str_t s1, str_t s2, const HamDev& H) {
    const int L = H.L;
    const str_t com = s1 & s2, a = s1 & ~s2, b = s2 & ~s1;
    const int a0 = __builtin_ctzll(a), a1 = 63 - __builtin_clzll(a);
    const int b0 = __builtin_ctzll(b), b1 = 63 - __builtin_clzll(b);
    const int diff = stacked(com, a0, a1) + stacked(com, b0, b1);
    const double e = H.V[(((size_t)a0 * L + a1) * L + b0) * L + b1] - H.V[(((size_t)a0 * L + a1) * L + b1) * L + b0];
    return (diff & 1) ? -e : e;
}

// Connections of each string, one wavefront per string, all pairs.
template <bool FILL>
__global__ void __launch_bounds__(256) k_det_conn(uint64_t n, const uint64_t* __restrict__ s, HamDev H,
                                                  uint32_t* __restrict__ cnt, uint32_t* __restrict__ scnt,
                                                  const int64_t* __restrict__ off, const int64_t* __restrict__ soff,
                                                  DetConn* __restrict__ conn, DetConn* __restrict__ sub,
                                                  double* __restrict__ d1) {
    const int lane = threadIdx.x & 63;
    const uint64_t I = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (I >= n) return;
    const str_t si = s[I];
    uint32_t c = 0, sc = 0;
    for (uint64_t j0 = 0; j0 < n; j0 += 64) {
        const uint64_t j = j0 + lane;
        const str_t sj = j < n ? s[j] : 0;
        const int d = j < n ? __popcll(si ^ sj) : 64;
        const uint64_t m = __ballot(d <= 4), ms = __ballot(d <= 2);
        if (FILL && d <= 4) {
            DetConn x;
            x.J = (uint32_t)j;
            x.type = (uint8_t)(d / 2);
            x.sign = 1;
            x.f = x.t = 0;
            x.x = x.xr = 0.0;
            if (d == 2) {  // one_diff_orbital without the other spin (CIMethod.cpp:409-427)
                const int L = H.L;
                const str_t com = si & sj;
                const int f = __builtin_ctzll(si & ~sj), t = __builtin_ctzll(sj & ~si);
                const int p = f < t ? f : t, q = f < t ? t : f;
                double e = H.h[p * L + q];
                for (str_t u = com; u; u &= u - 1) {
                    const int z = __builtin_ctzll(u);
                    e += H.V[(((size_t)p * L + z) * L + q) * L + z] - H.V[(((size_t)p * L + z) * L + z) * L + q];
                }
                x.f = (uint8_t)f;
                x.t = (uint8_t)t;
                x.sign = (stacked(com, p, q) & 1) ? -1 : 1;
                x.x = e;
            } else if (d == 4) {
                x.x = two_same(si, sj, H);
                x.xr = two_same(sj, si, H);
            }
            conn[off[I] + c + lanes_below(m)] = x;
            if (d <= 2) sub[soff[I] + sc + lanes_below(ms)] = x;
        }
        c += (uint32_t)__popcll(m);
        sc += (uint32_t)__popcll(ms);
    }
    if (lane == 0) {
        if (FILL) {
            d1[I] = diag_one_string(si, H);
        } else {
            cnt[I] = c;
            scnt[I] = sc;
        }
    }
}

struct TabArgs {
    const uint64_t *sa, *sb;
    const double *d1a, *d1b;
    const int64_t *offa, *offb, *soffb;
    const DetConn *conna, *connb, *subb;
    uint64_t nb;
    const uint32_t *ia, *ib, *pos;
};

// One wavefront per row.  Alpha connections are taken 64 at a time, one a lane;
// the scan of their beta counts spreads their candidates over the lanes in
// ascending order.
template <bool FILL>
__global__ void __launch_bounds__(256) k_det_rows_tab(TabArgs T, DetRowsArgs a) {
    __shared__ uint32_t pre[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint64_t i = (uint64_t)blockIdx.x * 4 + w;
    if (i >= a.n) return;  // a whole wavefront; no barrier follows
    const HamDev& H = a.H;
    const int L = H.L;
    const uint32_t ua = T.ia[i], ub = T.ib[i];
    const str_t Su = T.sa[ua], Sd = T.sb[ub];
    const int64_t a0 = T.offa[ua], an = T.offa[ua + 1] - a0;
    const DetConn* cb = T.connb + T.offb[ub];
    const uint32_t nb = (uint32_t)(T.offb[ub + 1] - T.offb[ub]);
    const DetConn* sb = T.subb + T.soffb[ub];
    const uint32_t nsb = (uint32_t)(T.soffb[ub + 1] - T.soffb[ub]);
    const int64_t base = FILL ? a.rowptr[i] : 0;
    uint32_t cnt = 0;
    volatile uint32_t* pw = pre[w];
    for (int64_t e0 = 0; e0 < an; e0 += 64) {
        const int type = e0 + lane < an ? T.conna[a0 + e0 + lane].type : 3;
        const uint32_t len = type == 0 ? nb : type == 1 ? nsb : type == 2 ? 1u : 0u;
        uint32_t inc = len;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t v = __shfl_up(inc, o, 64);
            if (lane >= o) inc += v;
        }
        __builtin_amdgcn_wave_barrier();  // the last batch has been read
        pw[lane] = inc - len;
        __builtin_amdgcn_wave_barrier();
        const uint32_t total = __shfl(inc, 63, 64);
        for (uint32_t t0 = 0; t0 < total; t0 += 64) {
            const uint32_t t = t0 + lane;
            bool keep = false;
            uint32_t j = 0;
            double v = 0.0;
            if (t < total) {
                int q = 0;  // the last entry that begins at or before t (empty ones follow the others)
#pragma unroll
                for (int step = 32; step > 0; step >>= 1)
                    if (pw[q + step] <= t && q + step < 64) q += step;
                // entries past the list have length 0 and begin at total > t
                const DetConn ea = T.conna[a0 + e0 + q];
                const uint32_t u = t - pw[q];
                DetConn eb;
                if (ea.type == 0) eb = cb[u];
                else if (ea.type == 1) eb = sb[u];
                else eb.J = ub, eb.type = 0;
                j = T.pos[(uint64_t)ea.J * T.nb + eb.J];
                if (j != 0xffffffffu) {
                    const bool first = j >= i;  // this row's determinant first
                    if (ea.type == 0) {
                        if (eb.type == 0) {  // diagonal (CIMethod.cpp:398-407)
                            v = T.d1a[ua];
                            v += T.d1b[ub];
                            v += jmix(Su, Sd, H);
                        } else if (eb.type == 1) {
                            const int p = eb.f < eb.t ? eb.f : eb.t, r = eb.f < eb.t ? eb.t : eb.f;
                            const double* wr = H.W + ((size_t)p * L + r) * L;
                            v = eb.x;
                            for (str_t s = Su; s; s &= s - 1) v += wr[__builtin_ctzll(s)];
                            if (eb.sign < 0) v = -v;
                        } else {
                            v = first ? eb.x : eb.xr;
                        }
                    } else if (ea.type == 1) {
                        if (eb.type == 0) {
                            const int p = ea.f < ea.t ? ea.f : ea.t, r = ea.f < ea.t ? ea.t : ea.f;
                            const double* wr = H.W + ((size_t)p * L + r) * L;
                            v = ea.x;
                            for (str_t s = Sd; s; s &= s - 1) v += wr[__builtin_ctzll(s)];
                            if (ea.sign < 0) v = -v;
                        } else {
                            const size_t i0 = first ? ea.f : ea.t, i1 = first ? eb.f : eb.t;
                            const size_t i2 = first ? ea.t : ea.f, i3 = first ? eb.t : eb.f;
                            v = H.V[((i0 * L + i1) * L + i2) * L + i3];
                            if (ea.sign != eb.sign) v = -v;
                        }
                    } else {
                        v = first ? ea.x : ea.xr;
                    }
                    keep = fabs(v) > a.zero;
                }
            }
            const uint64_t mask = __ballot(keep);
            if (FILL && keep) {
                const int64_t at = base + cnt + lanes_below(mask);
                a.col[at] = j;
                a.val[at] = v;
                if (a.val32) a.val32[at] = (float)v;
            }
            cnt += (uint32_t)__popcll(mask);
        }
    }
    if (!FILL && lane == 0) a.rowcnt[i] = cnt;
}

unsigned blocks(uint64_t n) { return (unsigned)((n + 255) / 256); }

// Distinct values of key >> shift (key sorted) into S; false if more than `most`.
bool distinct(DetStrings& S, uint64_t n, const uint64_t* key, int shift, uint64_t most, unsigned int* dup,
              hipStream_t st) {
    DBuf<uint32_t> first(n);
    DBuf<int64_t> at(n + 1);
    k_first<<<blocks(n), 256, 0, st>>>(n, key, shift, first.p, dup);
    CF_HIP(hipGetLastError());
    exclusive_scan_u32_to_i64(first.p, at.p, n, st);
    int64_t m = 0;
    CF_HIP(hipMemcpyAsync(&m, at.p + n, sizeof(m), hipMemcpyDeviceToHost, st));
    CF_HIP(hipStreamSynchronize(st));
    S.n = (uint64_t)m;
    if (S.n > most) return false;
    S.s.alloc(S.n);
    k_strings_of<<<blocks(n), 256, 0, st>>>(n, key, shift, first.p, at.p, S.s.p);
    CF_HIP(hipGetLastError());
    return true;
}

void connect(DetStrings& S, HamDev H, hipStream_t st) {
    DBuf<uint32_t> cnt(S.n), scnt(S.n);
    S.off.alloc(S.n + 1);
    S.soff.alloc(S.n + 1);
    S.d1.alloc(S.n);
    const unsigned grid = (unsigned)((S.n + 3) / 4);
    k_det_conn<false><<<grid, 256, 0, st>>>(S.n, S.s.p, H, cnt.p, scnt.p, nullptr, nullptr, nullptr, nullptr, nullptr);
    CF_HIP(hipGetLastError());
    exclusive_scan_u32_to_i64(cnt.p, S.off.p, S.n, st);
    exclusive_scan_u32_to_i64(scnt.p, S.soff.p, S.n, st);
    int64_t tot[2];
    CF_HIP(hipMemcpyAsync(&tot[0], S.off.p + S.n, sizeof(int64_t), hipMemcpyDeviceToHost, st));
    CF_HIP(hipMemcpyAsync(&tot[1], S.soff.p + S.n, sizeof(int64_t), hipMemcpyDeviceToHost, st));
    CF_HIP(hipStreamSynchronize(st));
    S.conn.alloc((uint64_t)tot[0]);
    S.sub.alloc((uint64_t)tot[1]);
    k_det_conn<true><<<grid, 256, 0, st>>>(S.n, S.s.p, H, nullptr, nullptr, S.off.p, S.soff.p, S.conn.p, S.sub.p,
                                           S.d1.p);
    CF_HIP(hipGetLastError());
}

}  // namespace

bool make_det_tables(DetTables& T, uint64_t n, const str_t* up, const str_t* down, const uint64_t* skey, HamDev H,
                     hipStream_t st) {
    constexpr uint64_t kMost = 16384;
    if (!n || n > 0x7fffffffull) return false;
    DBuf<unsigned int> dup(1);
    k_fill_u32<<<1, 256, 0, st>>>(1, 0u, dup.p);
    CF_HIP(hipGetLastError());
    if (!distinct(T.a, n, skey, 32, std::min(kMost, n), dup.p, st)) return false;
    unsigned int hdup = 0;
    CF_HIP(hipMemcpyAsync(&hdup, dup.p, sizeof(hdup), hipMemcpyDeviceToHost, st));
    DBuf<uint64_t> dk(n), ds(n);
    k_narrow_down<<<blocks(n), 256, 0, st>>>(n, skey, dk.p);
    CF_HIP(hipGetLastError());
    size_t tb = 0;
    CF_HIP(hipcub::DeviceRadixSort::SortKeys(nullptr, tb, dk.p, ds.p, (int)n, 0, H.L, st));
    DBuf<unsigned char> tmp(tb ? tb : 1);
    CF_HIP(hipcub::DeviceRadixSort::SortKeys(tmp.p, tb, dk.p, ds.p, (int)n, 0, H.L, st));
    if (!distinct(T.b, n, ds.p, 0, kMost, nullptr, st)) return false;  // waits for hdup too
    if (hdup || T.a.n * T.b.n > (n < 4096 ? 8 : 32) * n) return false;
    connect(T.a, H, st);
    connect(T.b, H, st);
    T.n = n;
    T.ia.alloc(n);
    T.ib.alloc(n);
    const uint64_t np = T.a.n * T.b.n;
    T.pos.alloc(np);
    k_fill_u32<<<blocks(np), 256, 0, st>>>(np, 0xffffffffu, T.pos.p);
    CF_HIP(hipGetLastError());
    k_det_index<<<blocks(n), 256, 0, st>>>(n, up, down, T.a.s.p, T.a.n, T.b.s.p, T.b.n, T.ia.p, T.ib.p, T.pos.p);
    CF_HIP(hipGetLastError());
    return true;
}

void launch_det_rows_tab(const DetTables& T, const DetRowsArgs& r, bool fill, hipStream_t st) {
    TabArgs a;
    a.sa = T.a.s.p;
    a.sb = T.b.s.p;
    a.d1a = T.a.d1.p;
    a.d1b = T.b.d1.p;
    a.offa = T.a.off.p;
    a.offb = T.b.off.p;
    a.soffb = T.b.soff.p;
    a.conna = T.a.conn.p;
    a.connb = T.b.conn.p;
    a.subb = T.b.sub.p;
    a.nb = T.b.n;
    a.ia = T.ia.p;
    a.ib = T.ib.p;
    a.pos = T.pos.p;
    const unsigned grid = (unsigned)((r.n + 3) / 4);
    if (fill) k_det_rows_tab<true><<<grid, 256, 0, st>>>(a, r);
    else k_det_rows_tab<false><<<grid, 256, 0, st>>>(a, r);
    CF_HIP(hipGetLastError());
}

}  // namespace cf
