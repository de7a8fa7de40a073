// nested1.h -- gfx950 passes of up to four right-hand sides with a nested far
// field (templates; instantiated per rank bucket, ranks up to 32, by inst_r*.hip).
//
// Per level, every point enters the moments of each cluster above it and every
// row evaluates each covering cluster's series (12 levels at n = 2^20). Here a
// point enters its tree leaf's moments alone and a row evaluates its leaf's
// series alone; the interval trees carry the rest by the two fixed
// re-expansion matrices of a half (T_k(s/2 -+ 1/2) = sum_m M[k][m] T_m(s)).
// Each side's tree is cut at plan time into subtrees of a few chunks (N1Sub);
// one workgroup walks a subtree in LDS, and the part of the tree above it as a
// path of single nodes, so a product is three launches:
//   up         per subtree: its leaves' moments, mu_P = M_0 mu_0 + M_1 mu_1 up
//              to its root, w = A mu of the clusters in it; then the root's
//              moments re-expanded up the path, one slot per cluster met
//   translate  per cluster of the output side: z = sum_b F_b w_b; a source above
//              the subtrees is summed from its slots (in slot order);
//              coefficients c = A^T z (w and z with the node offsets, N1Mat)
//   down       per subtree: coefficients down the path and the subtree by one
//              wavefront, then one series per row, added onto y
// The near field, y = beta*y + near, needs nothing of the chain and fills the
// first two launches, which wait on latencies. No atomics; the order of every
// sum is fixed by the plan.
//
// Few chunks: a near workgroup takes one, its columns (read by scalar loads)
// split over the wavefronts. Many: a wavefront takes two chunks, a row of each
// per lane, and its columns through LDS. (By scalar loads throughout, n = 2^20
// took 127 us, waiting on the scalar caches: 1.7 M 64-byte requests, four of
// five misses.)
//
// Two to four right-hand sides share a launch: an entry of the near field and of
// F is formed (or read) once for them, and a wavefront per right-hand side walks
// the tree. Single products four times over would form the entries four times;
// the per-level passes read every level's U, V and F once for four.
//
// Measured (FP64, n = 2^20, leaf 256, rank 24, Cauchy): stored 1237 -> 178 us
// a product, matrix-free 236 -> 128 us, where the vector instructions alone
// take 62 us (near) and 17 us (far); transposed stored, n = 200003, leaf 80,
// rank 20: 432 -> 62 us; Float32 hybrid, n = 500009, rank 10: 180 -> 63 us;
// n = 1000: 25.9 -> 22.2 us. Four right-hand sides, stored log kernel, n = 2^17,
// leaf 80, rank 20: 349 -> 151 us (the translation, whose log entries of F and
// of the near field are read, takes 66 of them, the upward pass 57).
#pragma once
#include "kernels_impl.h"

namespace hmxk {
namespace {

// Where the near field's entries and F come from:
// (N1_FREE, N1_EXACT and N1_READ of hmx_device.h)
//   N1_FREE   formed from the points and nodes, several terms of 1/d^m on one
//             reciprocal (matrix-free products)
//   N1_EXACT  formed term by term, as the stored entries are rounded, and summed
//             in the order of N1_READ: a stored or hybrid plan of 1/d^m, whose
//             values it saves reading. New points may bring entries that the
//             refined reciprocal does not give (points that meet, distances out
//             of range): the plan's word odd[1], written with the entries and
//             read here, then has every value formed by division. So the route
//             hangs on nothing that the host would have to wait for, and a
//             captured product holds for later points too.
//   N1_READ   the stored entries (the log kernel, a caller's f, entries that
//             are not all finite)

// ----------------------------------------------------- wave-uniform loads
template <class T> struct Vec8;
template <> struct Vec8<double> { typedef double type __attribute__((ext_vector_type(8), aligned(8))); };
template <> struct Vec8<float> { typedef float type __attribute__((ext_vector_type(8), aligned(4))); };
#define HMX_CONST_AS __attribute__((address_space(4)))

// o = p[0 .. 7] by scalar loads (p wave-uniform, not written by this kernel)
template <class T>
__device__ __forceinline__ void sload8(const T *p, T (&o)[8]) {
    using V = typename Vec8<T>::type;
    const V v = *(const HMX_CONST_AS V *)(p);
#pragma unroll
    for (int u = 0; u < 8; ++u) o[u] = v[u];
}
template <class T> struct Vec4;
template <> struct Vec4<double> { typedef double type __attribute__((ext_vector_type(4), aligned(8))); };
template <> struct Vec4<float> { typedef float type __attribute__((ext_vector_type(4), aligned(4))); };
template <class T>
__device__ __forceinline__ void sload4(const T *p, T (&o)[4]) {
    using V = typename Vec4<T>::type;
    const V v = *(const HMX_CONST_AS V *)(p);
#pragma unroll
    for (int u = 0; u < 4; ++u) o[u] = v[u];
}
template <class T>
__device__ __forceinline__ T sload1(const T *p) {
    return *(const HMX_CONST_AS T *)(p);
}

// a table record (a multiple of 4 bytes) by scalar loads
template <class S>
__device__ __forceinline__ S sload_struct(const S *p) {
    constexpr int N = sizeof(S) / 4;
    int32_t w[N];
    const HMX_CONST_AS int32_t *q = (const HMX_CONST_AS int32_t *)(const void *)p;
#pragma unroll
    for (int k = 0; k < N; ++k) w[k] = q[k];
    S o;
    __builtin_memcpy(&o, w, sizeof(S));
    return o;
}

// ------------------------------------------------------------- near field
// zero, denormal, infinity or NaN
__device__ __forceinline__ bool odd_class(double v) { return __builtin_amdgcn_class(v, 0x2F7); }
__device__ __forceinline__ bool odd_class(float v) { return __builtin_amdgcn_classf(v, 0x2F7); }
__device__ __forceinline__ double rcp_raw(double v) { return __builtin_amdgcn_rcp(v); }
__device__ __forceinline__ float rcp_raw(float v) { return __builtin_amdgcn_rcpf(v); }
__device__ __forceinline__ double rcp_refine(double d, double r) {
    double e = __builtin_fma(-d, r, 1.0);
    r = __builtin_fma(r, e, r);
    e = __builtin_fma(-d, r, 1.0);
    return __builtin_fma(r, e, r);
}
__device__ __forceinline__ float rcp_refine(float d, float r) {
    const float e = __builtin_fmaf(-d, r, 1.0f);
    return __builtin_fmaf(r, e, r);
}

// acc_i + sum_{u < N} f(p_i, q_u) v_u for NR rows (f(q_u, p_i) when TR).
// 1/d^m: four columns share the reciprocal of their denominators' product, and
// each pair's is taken out of it, 1/(d0 d1) = d2 d3 / (d0 d1 d2 d3), before it
// meets the inputs: v0/d0 + v1/d1 = (v0 d1 + v1 d0) / (d0 d1), a numerator of
// v d. (Over one common denominator it is v d^3, which leaves the range where
// every term lies within it: Float32 inputs of 1e-28 at n = 2^20 lost 5 %.) FP32,
// whose range v d leaves too, takes each term's own reciprocal, d1 / (d0 d1); its
// d^2 and d^3 share one between two columns only. If a reciprocal (FP32: or a
// denominator) leaves the normal range (zero, denormal, infinite or NaN) it
// returns true, and the caller forms its sum again from where it began, term by
// term (near_single). No branch between the columns, whose chains then run side
// by side: a branch for each four took 45 us more at n = 2^20, one for each
// eight 4. n = 2^20, leaf 256, rank 24: Cauchy 125 us, Coulomb 138 (common
// denominator 126 and 140); Float32, leaf 64, rank 16: 96 us (90).
// EXACT: term by term. The reciprocal's last step starts within 2^-48 (FP32
// 2^-22) of it, so the result is a division's but for rare half-way cases
// (<= 1 ulp).
// log: columns outside lo <= u < hi are padding, which adds nothing (a repeated
// column that meets the row's point has an infinite value).
template <class T, int KID, bool TR, bool EXACT, int N, int NR>
__device__ __forceinline__ bool near_terms(const T *p, const T *q, const T *v, T *acc, int lo,
                                           int hi) {
    bool odd = false;
    if constexpr (KID <= 2 && !EXACT) {
        constexpr int S = (sizeof(T) == 8 || KID == 0) ? 4 : 2, G = N / S;
        auto dist = [&](int i, int u) {
            const T e = TR ? q[u] - p[i] : p[i] - q[u];
            return KID == 0 ? e : KID == 1 ? e * e : e * e * e;
        };
        // v0/d0 + v1/d1 added on, r = 1/(d0 d1)
        auto pair = [&](int i, int u, T r, T d0, T d1) {
            if constexpr (sizeof(T) == 8) {
                acc[i] = fmaT(fmaT(v[u], d1, v[u + 1] * d0), r, acc[i]);
            } else {
                acc[i] = fmaT(r * d1, v[u], acc[i]);
                acc[i] = fmaT(r * d0, v[u + 1], acc[i]);
            }
        };
        auto test = [&](T r, T a, T b) {
            odd |= odd_class(r);
            if constexpr (sizeof(T) == 4) {
                odd |= odd_class(a);
                odd |= odd_class(b);
            }
        };
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                const int u = g * S;
                const T d0 = dist(i, u), d1 = dist(i, u + 1), a = d0 * d1;
                if constexpr (S == 4) {
                    const T d2 = dist(i, u + 2), d3 = dist(i, u + 3), b = d2 * d3;
                    const T r0 = rcp_raw(a * b), r = rcp_refine(a * b, r0);
                    test(r0, a, b);
                    pair(i, u, r * b, d0, d1);
                    pair(i, u + 2, r * a, d2, d3);
                } else {
                    const T r0 = rcp_raw(a);
                    test(r0, a, a);
                    pair(i, u, rcp_refine(a, r0), d0, d1);
                }
            }
    } else {
#pragma unroll
        for (int u = 0; u < N; ++u)
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                const T f = TR ? kern_fast<T, KID>(q[u], p[i]) : kern_fast<T, KID>(p[i], q[u]);
                const T t = fmaT(f, v[u], acc[i]);
                acc[i] = KID <= 2 || (u >= lo && u < hi) ? t : acc[i];
            }
    }
    return odd;
}

// acc[i][k] + sum_u f(p_i, q_u) v[u][k] over the columns n0 <= u < n1 that
// col(u, q, v) reads, each value of 1/d^m a division of its own
template <class T, int KID, bool TR, int NR, int KB, class Col>
__device__ __forceinline__ void near_single(const T *p, int n0, int n1, Col col, T (*acc)[KB]) {
#pragma unroll 1
    for (int u = n0; u < n1; ++u) {
        T q, v[KB];
        col(u, q, v);
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const T d = TR ? q - p[i] : p[i] - q;
            const T f = T(1) / (KID == 0 ? d : KID == 1 ? d * d : d * d * d);
#pragma unroll
            for (int k = 0; k < KB; ++k) acc[i][k] = fmaT(f, v[k], acc[i][k]);
        }
    }
}

// acc[i][k] + sum_{u < N} f(p_i, q_u) v[u][k]: each value formed once for its KB
// right-hand sides (term by term: a shared reciprocal's numerators would be
// formed for each of them)
template <class T, int KID, bool TR, int N, int NR, int KB>
__device__ __forceinline__ void near_terms_kb(const T *p, const T *q, const T (*v)[KB],
                                              T (*acc)[KB], int lo, int hi) {
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const T f = TR ? kern_fast<T, KID>(q[u], p[i]) : kern_fast<T, KID>(p[i], q[u]);
#pragma unroll
            for (int k = 0; k < KB; ++k) {
                const T t = fmaT(f, v[u][k], acc[i][k]);
                acc[i][k] = KID <= 2 || (u >= lo && u < hi) ? t : acc[i][k];
            }
        }
}

// One row's sums over a chunk's dense blocks (its runs), N columns at a time:
// batches b0, b0 + bs, ... of each block. A block's last batch is its last N
// columns, those of the batch before it at weight zero; a block narrower than N
// repeats its last column at weight zero. (The next batch is not loaded ahead:
// two batches and the addresses do not fit the scalar registers, and the other
// wavefronts cover the loads.) row: the lane's row of the chunk. Of the KB
// right-hand sides, nq are there; the others repeat the last.
template <class T, int KID, bool TR, int SRC, int KB>
__device__ __forceinline__ void near_runs(const N1Run *runs, int nrun, T p, const T *pts_in,
                                          const T *A, const T *x, int64_t incx, int64_t ldx, int nq,
                                          int row, int b0, int bs, bool single, T (&acc)[KB]) {
    constexpr int N = KB == 1 ? 8 : 4;
#pragma unroll
    for (int k = 0; k < KB; ++k) acc[k] = T(0);
    for (int e = 0; e < nrun; ++e) {
        const N1Run R = sload_struct(runs + e);
        const T *qs = pts_in + R.q0, *vs = x + R.q0 * incx;
        // stored entries: element (row, j) of the block, tiles of 64 rows
        const int i = R.off + row;
        const T *Ar = SRC != N1_READ ? nullptr
                      : TR           ? A + R.aoff + (int64_t)i * HM_TILE
                                     : A + R.aoff + tile_index(i, 0, R.cols);
        auto entry = [&](int j) {
            return TR ? Ar[(int64_t)(j >> 6) * HM_TILE * R.cols + (j & (HM_TILE - 1))]
                      : Ar[j * HM_TILE];
        };
        T acc0[1][KB];
#pragma unroll
        for (int k = 0; k < KB; ++k) acc0[0][k] = acc[k];
        bool odd = single;
        for (int t = b0; N * t < R.n && !single; t += bs) {
            T q[N], v[N][KB];
            const int j0 = R.n >= N ? min(N * t, R.n - N) : 0;
            if (KB == 1 && R.n >= N && incx == 1) {
                if constexpr (KB == 1) {
                    T v8[8];
                    sload8(vs + j0, v8);
#pragma unroll
                    for (int u = 0; u < N; ++u) v[u][0] = v8[u];
                }
            } else if (KB == 4 && ldx == 1 && nq == 4) {
                if constexpr (KB == 4) {  // a row of x in one load
#pragma unroll
                    for (int u = 0; u < N; ++u) sload4(vs + min(j0 + u, R.n - 1) * incx, v[u]);
                }
            } else {
#pragma unroll
                for (int u = 0; u < N; ++u) {
                    const T *vj = vs + min(j0 + u, R.n - 1) * incx;
#pragma unroll
                    for (int k = 0; k < KB; ++k) v[u][k] = sload1(vj + min(k, nq - 1) * ldx);
                }
            }
            if (j0 < N * t || j0 + N > R.n) {
#pragma unroll
                for (int u = 0; u < N; ++u)
#pragma unroll
                    for (int k = 0; k < KB; ++k)
                        v[u][k] = j0 + u < N * t || j0 + u >= R.n ? T(0) : v[u][k];
            }
            if constexpr (SRC == N1_READ) {
#pragma unroll
                for (int u = 0; u < N; ++u) q[u] = entry(min(j0 + u, R.n - 1));
                // a column at weight zero adds nothing, whatever its entry
#pragma unroll
                for (int u = 0; u < N; ++u)
                    if (j0 + u >= N * t && j0 + u < R.n)
#pragma unroll
                        for (int k = 0; k < KB; ++k) acc[k] = fmaT(q[u], v[u][k], acc[k]);
            } else {
                if (KB == 1 && R.n >= N) {
                    if constexpr (KB == 1) sload8(qs + j0, q);
                } else {
#pragma unroll
                    for (int u = 0; u < N; ++u) q[u] = sload1(qs + min(j0 + u, R.n - 1));
                }
                if constexpr (KB == 1) {
                    T w[N];
#pragma unroll
                    for (int u = 0; u < N; ++u) w[u] = v[u][0];
                    odd |= near_terms<T, KID, TR, SRC == N1_EXACT, N, 1>(&p, q, w, acc, N * t - j0,
                                                                         R.n - j0);
                } else {
                    near_terms_kb<T, KID, TR, N, 1, KB>(&p, q, v, &acc, N * t - j0, R.n - j0);
                }
            }
        }
        if constexpr (KID <= 2 && SRC != N1_READ) {
            if (__builtin_expect(odd, 0)) {
                for (int t = b0; N * t < R.n; t += bs)
                    near_single<T, KID, TR, 1, KB>(&p, N * t, min(N * t + N, R.n),
                                                   [&](int u, T &qu, T (&vu)[KB]) {
                                                       qu = qs[u];
#pragma unroll
                                                       for (int k = 0; k < KB; ++k)
                                                           vu[k] = vs[u * incx + min(k, nq - 1) * ldx];
                                                   },
                                                   acc0);
#pragma unroll
                for (int k = 0; k < KB; ++k) acc[k] = acc0[0][k];
            }
        }
    }
}

// Columns in LDS, for wavefronts with two rows per lane (rows of two chunks):
// a point and its KB inputs. A 16-byte broadcast read takes 8 LDS cycles, shared
// by four SIMDs, where a row's four terms take 23 vector cycles a column: read
// for one row alone, LDS would be the slower of the two.
template <class T, int KB>
struct NearCol {
    T q, v[KB];
};

// the sums of a tile's n columns (padded at weight zero to a multiple of eight)
// for one or both rows
template <class T, int KID, bool TR, bool EXACT, int NR, int KB>
__device__ __forceinline__ void near_tile(const NearCol<T, KB> *t, int n, const T (&p)[NR],
                                          bool single, T (&acc)[NR][KB]) {
    constexpr int N = KID == 3 || KB > 1 ? 2 : 8;
    T acc0[NR][KB];
    bool odd = single;
#pragma unroll
    for (int i = 0; i < NR; ++i)
#pragma unroll
        for (int k = 0; k < KB; ++k) acc0[i][k] = acc[i][k];
    for (int j = 0; j < n && !single; j += N) {
        T q[N], v[N][KB];
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const NearCol<T, KB> c = t[j + u];
            q[u] = c.q;
#pragma unroll
            for (int k = 0; k < KB; ++k) v[u][k] = c.v[k];
        }
        if constexpr (KB == 1) {
            T w[N], s[NR];
#pragma unroll
            for (int u = 0; u < N; ++u) w[u] = v[u][0];
#pragma unroll
            for (int i = 0; i < NR; ++i) s[i] = acc[i][0];
            odd |= near_terms<T, KID, TR, EXACT, N, NR>(p, q, w, s, 0, n - j);
#pragma unroll
            for (int i = 0; i < NR; ++i) acc[i][0] = s[i];
        } else {
            near_terms_kb<T, KID, TR, N, NR, KB>(p, q, v, acc, 0, n - j);
        }
    }
    if constexpr (KID <= 2) {
        if (__builtin_expect(odd, 0)) {
            near_single<T, KID, TR, NR, KB>(p, 0, n, [&](int u, T &qu, T (&vu)[KB]) {
                qu = t[u].q;
#pragma unroll
                for (int k = 0; k < KB; ++k) vu[k] = t[u].v[k];
            }, acc0);
#pragma unroll
            for (int i = 0; i < NR; ++i)
#pragma unroll
                for (int k = 0; k < KB; ++k) acc[i][k] = acc0[i][k];
        }
    }
}

// Near field of a unit (one or two chunks, a row of each per lane): its runs'
// columns pass through this wavefront's LDS 64 at a time, the next tile's
// loads in flight meanwhile. A run serves the first chunk (mask 1), the second
// (2) or both (3).
template <class T, int KID, bool TR, bool EXACT, int KB>
__device__ __forceinline__ void near_unit(const N1UnitRun *runs, int nrun, const T (&p)[2],
                                          const T *pts_in, const T *x, int64_t incx, int64_t ldx,
                                          int nq, NearCol<T, KB> (*tile)[WAVE], int lane,
                                          bool single, T (&acc)[2][KB]) {
    if (nrun == 0) return;
    N1UnitRun R = sload_struct(runs);
    int e = 0, j = 0, b = 0;
    auto load = [&](const N1UnitRun &Q, int j0, NearCol<T, KB> &c) {
        const int64_t at = Q.q0 + min(j0 + lane, Q.n - 1);
        c.q = pts_in[at];
#pragma unroll
        for (int k = 0; k < KB; ++k) c.v[k] = x[at * incx + min(k, nq - 1) * ldx];
    };
    NearCol<T, KB> c;
    load(R, 0, c);
    while (e < nrun) {
        const int n = min(WAVE, R.n - j), mask = R.mask;
        if (lane >= n) {
#pragma unroll
            for (int k = 0; k < KB; ++k) c.v[k] = T(0);
        }
        NearCol<T, KB> *t = tile[b];
        t[lane] = c;
        wave_sync();
        j += WAVE;
        if (j >= R.n) {
            j = 0;
            if (++e < nrun) R = sload_struct(runs + e);
        }
        if (e < nrun) load(R, j, c);
        if (mask == 3) {
            near_tile<T, KID, TR, EXACT, 2, KB>(t, n, p, single, acc);
        } else {
            const T p1[1] = {mask == 1 ? p[0] : p[1]};
            T a1[1][KB];
#pragma unroll
            for (int k = 0; k < KB; ++k) a1[0][k] = mask == 1 ? acc[0][k] : acc[1][k];
            near_tile<T, KID, TR, EXACT, 1, KB>(t, n, p1, single, a1);
#pragma unroll
            for (int k = 0; k < KB; ++k) {
                if (mask == 1) acc[0][k] = a1[0][k];
                else acc[1][k] = a1[0][k];
            }
        }
        b ^= 1;
    }
}

template <class T>
__device__ __forceinline__ void n1_write(const N1Chunk &C, const MvArgsT<T> &a, int q, int beta,
                                         int lane, T v) {
    if (lane < C.np) {
        T *yo = a.y + (C.p0 + lane) * a.incy + q * a.ldy;
        *yo = (beta ? *yo : T(0)) + v;
    }
}

// One workgroup of the near field, y = beta*y + near: a chunk, its columns
// split over the wavefronts and their sums added in LDS in wavefront order, or
// (with units) a unit per wavefront.
template <class T, int KB>
struct NearLds {
    union {
        NearCol<T, KB> tile[WPB][2][WAVE];
        T red[WPB][KB][WAVE];
    };
    __device__ NearLds() {}
};
template <class T, int KID, bool TR, int SRC, int KB>
__device__ __forceinline__ void near_block(const N1Side &o, int blk, const T *pts_out,
                                           const T *pts_in, const T *A, const int32_t *odd,
                                           const MvArgsT<T> &a, int nq, NearLds<T, KB> &s) {
    const int lane = threadIdx.x % WAVE, wv = uniform((int)(threadIdx.x / WAVE));
    // an entry that the refinement does not give as it is stored: all by division
    const bool single = SRC == N1_EXACT && odd && odd[1] != 0;
    if (o.nunit == 0) {
        const N1Chunk C = sload_struct(o.ch + blk);
        const int row = min(lane, C.np - 1);
        const T po = SRC == N1_READ ? T(0) : pts_out[C.p0 + row];
        T acc[KB];
        near_runs<T, KID, TR, SRC, KB>(o.run + C.run, C.nrun, po, pts_in, A, a.x, a.incx, a.ldx, nq,
                                       row, wv, WPB, single, acc);
#pragma unroll
        for (int k = 0; k < KB; ++k) s.red[wv][k][lane] = acc[k];
        __syncthreads();
        // wavefront k adds right-hand side k's sums (KB <= WPB)
        if (wv >= min(KB, nq)) return;
        T v = s.red[0][wv][lane];
#pragma unroll
        for (int u = 1; u < WPB; ++u) v += s.red[u][wv][lane];
        n1_write(C, a, wv, a.beta, lane, v);
        return;
    }
    if constexpr (SRC == N1_READ) return;  // stored entries in units: k_down's near part
    const int c = blk * WPB + wv;
    if (c >= o.nunit) return;
    const N1Unit Un = sload_struct(o.unit + c);
    N1Chunk C[2];
    T po[2], acc[2][KB];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        C[q] = sload_struct(o.ch + Un.ch + (q < Un.nch ? q : 0));
        po[q] = pts_out[C[q].p0 + min(lane, C[q].np - 1)];
#pragma unroll
        for (int k = 0; k < KB; ++k) acc[q][k] = T(0);
    }
    near_unit<T, KID, TR, SRC == N1_EXACT, KB>(o.urun + Un.run, Un.nrun, po, pts_in, a.x, a.incx,
                                               a.ldx, nq, s.tile[wv], lane, single, acc);
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int k = 0; k < KB; ++k)
            if (q < Un.nch && k < nq) n1_write(C[q], a, k, a.beta, lane, acc[q][k]);
}

// -------------------------------------------------------------- far field
// A plan's r x r matrices for lanes (m, h) = (lane % 32, lane / 32), padded
// with zeros to RMAX, one row of 64 values per step: M_h[m][k] and M_h[k][m] for
// k < RMAX, A[m][h' + j], A[h' + j][m], D[h' + j][m] and D[m][h' + j] for
// j < RMAX / 2, h' = h RMAX / 2.
//
// F holds f at the mapped nodes as they are rounded, up to 1e-12 of a half width
// off the exact ones (2^-53 of the point against a deep cluster). The products'
// polynomials go through the rounded nodes: their offsets d enter w and z to
// first order, w = w0 - D^T (d w0) for w0 = A mu, and c = A^T (z - d (D z)), D
// the differentiation matrix of the exact nodes (held at 2^-12 and d at 2^12
// times itself: D's entries reach r^2, and D z would leave the range before c
// does). Without it, stored products at
// n = 2^20 were 6.4e-15 off, and 1.3e-15 with U and V, which hold the basis at
// the rounded nodes.
template <class T, int RMAX>
struct N1Mat {
    static constexpr int HALF = RMAX / 2;
    static constexpr int MU = 0, MD = RMAX * WAVE, AU = 2 * RMAX * WAVE,
                         DU = AU + HALF * WAVE, AT = DU + HALF * WAVE, DD = AT + HALF * WAVE;
};
template <class T, int N>
__device__ __forceinline__ void load_rows(const T *m, int lane, T (&row)[N]) {
#pragma unroll
    for (int k = 0; k < N; ++k) row[k] = m[k * WAVE + lane];
}
// sum_k row[k] v[k], v in LDS (entries past r: finite, or the row's are zero)
template <class T, int N>
__device__ __forceinline__ T dot_row(const T (&row)[N], const T *v) {
    T s0 = T(0), s1 = T(0);
#pragma unroll
    for (int k = 0; k < N; k += 2) {
        s0 = fmaT(row[k], v[k], s0);
        s1 = fmaT(row[k + 1], v[k + 1], s1);
    }
    return s0 + s1;
}

// the same with the lane's column of rows of 64 in LDS
template <class T, int HALF>
__device__ __forceinline__ T dot_lds(const T *rows, int lane, const T *v) {
    T s0 = T(0), s1 = T(0);
#pragma unroll
    for (int k = 0; k < HALF; k += 2) {
        s0 = fmaT(rows[k * WAVE + lane], v[k], s0);
        s1 = fmaT(rows[(k + 1) * WAVE + lane], v[k + 1], s1);
    }
    return s0 + s1;
}

// The moments sum_j T_m(xh_j) x_j of one leaf's points (one wavefront)
template <class T, int RMAX>
__device__ __forceinline__ void leaf_moments(const N1Leaf &L, const T *pts, const T *x, int64_t incx,
                                             int lane, T *out) {
    const T cx = (T)L.f.cx, cl = (T)L.f.cl, cy = (T)L.f.cy;
    T acc[RMAX];
#pragma unroll
    for (int k = 0; k < RMAX; ++k) acc[k] = T(0);
    for (int i = lane; i < L.len; i += WAVE) {
        const T xv = x[(L.first + i) * incx];
        const T xh = ((pts[L.first + i] - cx) - cl) * cy;
        const T x2 = xh + xh;
        T t0 = xv, t1 = xh * xv;  // T_m(xh) x by the recurrence
        acc[0] += t0;
        acc[1] += t1;
#pragma unroll
        for (int k = 2; k < RMAX; ++k) {
            const T t2 = fmaT(x2, t1, -t0);
            acc[k] += t2;
            t0 = t1;
            t1 = t2;
        }
    }
    int base = 0;
    Halve<RMAX, WAVE / 2>::run(acc, lane, base);
    constexpr int LEFT = HalveShape<RMAX, WAVE / 2>::left;
    constexpr int MASK = HalveShape<RMAX, WAVE / 2>::mask;
    if ((lane & MASK) == 0) {
#pragma unroll
        for (int i = 0; i < LEFT; ++i) out[base + i] = acc[i];
    }
}

// One node's moments from its halves' (zero for an empty one)
template <class T, int RMAX>
__device__ __forceinline__ void node_moments(const N1Node &N, const T (&Mr)[RMAX], T (*mom)[RMAX],
                                             int n, int m, int h) {
    if (N.c[0] < 0 && N.c[1] < 0) return;  // a leaf (wave-uniform)
    const int c = h ? N.c[1] : N.c[0];
    T v = dot_row(Mr, mom[c >= 0 ? c : 0]);
    if (c < 0) v = T(0);
    v += __shfl_xor(v, 32);
    if (h == 0 && m < RMAX) mom[n][m] = v;
}

// The w of NB clusters from their moments mom (LDS), d the lane's node offsets,
// tmp: LDS of this wavefront's; dot_a and dot_d: the lane's row of A and of D^T
// times a vector in LDS. Together, so that their chains run side by side.
template <int RMAX, int NB, class T, class DotA, class DotD>
__device__ __forceinline__ void node_values(DotA dot_a, DotD dot_d, const T *const (&mom)[NB],
                                            const T (&d)[NB], int m, int h, T (*tmp)[RMAX],
                                            T (&v)[NB]) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        v[b] = dot_a(mom[b] + h * (RMAX / 2));
        v[b] += __shfl_xor(v[b], 32);
        if (h == 0 && m < RMAX) tmp[b][m] = d[b] * v[b];
    }
    wave_sync();
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        T e = dot_d(tmp[b] + h * (RMAX / 2));
        e += __shfl_xor(e, 32);
        v[b] -= e;
    }
    wave_sync();
}
// The w of a subtree's clusters, N1_WB at a time: of the local nodes next(-1),
// next(that), ... below nnode, cl(n) their clusters; put(cluster, k, w_k)
constexpr int N1_WB = 4;
template <int RMAX, class T, class Next, class Cl, class Put>
__device__ __forceinline__ void subtree_w(const T *mats, const T *del, const T (*mom)[RMAX],
                                          T (*tmp)[RMAX], int r, int nnode, int lane, Next next,
                                          Cl cl, Put put) {
    using Mt = N1Mat<T, RMAX>;
    const int m = lane & 31, h = lane >> 5;
    T Ar[Mt::HALF], Dr[Mt::HALF];
    load_rows(mats + Mt::AU, lane, Ar);
    load_rows(mats + Mt::DU, lane, Dr);
    for (int n = next(-1); n < nnode;) {
        const int first = n;
        int id[N1_WB];
        T d[N1_WB], v[N1_WB];
        const T *mo[N1_WB];
#pragma unroll
        for (int b = 0; b < N1_WB; ++b) {  // past the last: the first again, not written
            id[b] = n < nnode ? cl(n) : -1;
            mo[b] = mom[n < nnode ? n : first];
            d[b] = m < r ? del[(int64_t)(n < nnode ? id[b] : id[0]) * r + m] : T(0);
            if (n < nnode) n = next(n);
        }
        node_values<RMAX, N1_WB>([&](const T *u) { return dot_row(Ar, u); },
                                 [&](const T *u) { return dot_row(Dr, u); }, mo, d, m, h, tmp, v);
        if (h == 0 && m < r) {
#pragma unroll
            for (int b = 0; b < N1_WB; ++b)
                if (id[b] >= 0) put(id[b], m, v[b]);
        }
    }
}

// Upward pass, one workgroup per subtree of the input side. The subtree's
// records and the matrix rows are read before they are needed (the pass is a
// chain of latencies: a few leaves, the depths, the path).
template <class T, int RMAX>
struct UpLds {
    alignas(16) T mom[N1_NODES][RMAX];
    alignas(16) T pv[2][RMAX];
    alignas(16) T dw[WPB][N1_WB][RMAX];
    N1Node nodes[N1_NODES];
    int32_t lev[N1_NODES + 1];
};
template <class T, int RMAX>
__device__ __forceinline__ void n1_up_block(const N1Side &s, const T *pts, const T *x, int64_t incx,
                                            const T *mats, const T *del, T *partial, T *w, int r,
                                            int blk, UpLds<T, RMAX> &L_) {
    using Mt = N1Mat<T, RMAX>;
    auto &mom = L_.mom;
    auto &pv = L_.pv;
    auto &nodes = L_.nodes;
    auto &lev = L_.lev;
    const N1Sub S = sload_struct(s.sub + blk);
    const int lane = threadIdx.x % WAVE, wv = uniform((int)(threadIdx.x / WAVE));
    const int m = lane & 31, h = lane >> 5;
    if ((int)threadIdx.x < S.nnode) nodes[threadIdx.x] = s.node[S.node + threadIdx.x];
    if ((int)threadIdx.x <= S.nlev) lev[threadIdx.x] = s.lev[S.lev + threadIdx.x];
    // the path, its nodes' records in the lanes (the last wavefront walks it)
    int p_half = 0;
    int64_t p_slot = -1;
    if (wv == WPB - 1 && lane < min(S.npath, WAVE)) {
        const N1Path P = s.path[S.path + S.npath - 1 - lane];
        p_half = P.half;
        p_slot = P.slot;
    }
    for (int e = wv; e < S.nleaf; e += WPB) {
        const N1Leaf L = sload_struct(s.leaf + S.leaf + e);
        leaf_moments<T, RMAX>(L, pts, x, incx, lane, mom[L.loc]);
    }
    T Mr[RMAX];
    load_rows(mats + Mt::MU, lane, Mr);
    __syncthreads();
    for (int l = S.nlev - 2; l >= 0; --l) {
        const int nb = lev[l], ne = lev[l + 1];
        for (int n = nb + wv; n < ne; n += WPB) {
            node_moments<T, RMAX>(nodes[n], Mr, mom, n, m, h);
        }
        __syncthreads();
    }
    // w of the clusters; the last wavefront walks the path meanwhile
    if (wv < WPB - 1 || S.npath == 0) {
        const int step = S.npath == 0 ? WPB : WPB - 1;
        subtree_w<RMAX>(
            mats, del, mom, L_.dw[wv], r, S.nnode, lane,
            [&](int n) {
                n = n < 0 ? wv : n + step;
                while (n < S.nnode && nodes[n].cl < 0) n += step;
                return n;
            },
            [&](int n) { return nodes[n].cl; },
            [&](int cl, int k, T v) { w[(int64_t)cl * r + k] = v; });
        return;
    }
    const T *cur = mom[0];
    for (int e = 0; e < S.npath; ++e) {  // from the root's parent up
        if (e > 0 && e % WAVE == 0) {
            const int at = S.npath - 1 - e - lane;
            if (at >= 0) {
                const N1Path P = s.path[S.path + at];
                p_half = P.half;
                p_slot = P.slot;
            }
        }
        const int64_t slot = rl_l(p_slot, e % WAVE);
        T v = dot_row(Mr, cur);
        if (h != rl_i(p_half, e % WAVE)) v = T(0);
        v += __shfl_xor(v, 32);
        T *nx = pv[e & 1];
        if (h == 0 && m < RMAX) nx[m] = v;
        if (slot >= 0 && h == 0 && m < r) partial[slot * r + m] = v;
        wave_sync();
        cur = nx;
    }
}

// Upward pass of several right-hand sides: a wavefront takes one of them through
// the whole subtree, so that the wavefronts' chains of latencies run side by
// side without a barrier.
template <class T, int RMAX>
struct UpLdsKb {
    alignas(16) T mom[N1_KB][N1_NODES][RMAX];
    alignas(16) T pv[N1_KB][2][RMAX];
    alignas(16) T dw[N1_KB][N1_WB][RMAX];
};
template <class T, int RMAX>
__device__ __forceinline__ void n1_up_block_kb(const N1Side &s, const T *pts, const T *x,
                                               int64_t incx, int64_t ldx, const T *mats,
                                               const T *del, T *partial, T *w, int r, int nq,
                                               int blk, UpLdsKb<T, RMAX> &L_) {
    using Mt = N1Mat<T, RMAX>;
    static_assert(N1_KB == WPB, "a wavefront per right-hand side");
    const int lane = threadIdx.x % WAVE, q = uniform((int)(threadIdx.x / WAVE));
    if (q >= nq) return;
    const int m = lane & 31, h = lane >> 5;
    auto &mom = L_.mom[q];
    const N1Sub S = sload_struct(s.sub + blk);
    N1Node nd{-1, {-1, -1}};
    if (lane < S.nnode) nd = s.node[S.node + lane];
    int p_half = 0;
    int64_t p_slot = -1;
    auto load_path = [&](int e) {  // the path's nodes e + lane from the root's parent up
        const int at = S.npath - 1 - e - lane;
        if (at >= 0) {
            const N1Path P = s.path[S.path + at];
            p_half = P.half;
            p_slot = P.slot;
        }
    };
    load_path(0);
    x += q * ldx;
    for (int e = 0; e < S.nleaf; ++e) {
        const N1Leaf L = sload_struct(s.leaf + S.leaf + e);
        leaf_moments<T, RMAX>(L, pts, x, incx, lane, mom[L.loc]);
    }
    T Mr[RMAX];
    load_rows(mats + Mt::MU, lane, Mr);
    wave_sync();
    for (int n = S.nnode - 1; n >= 0; --n) {  // halves come after their node
        const N1Node N{0, {rl_i(nd.c[0], n), rl_i(nd.c[1], n)}};
        node_moments<T, RMAX>(N, Mr, mom, n, m, h);
        wave_sync();
    }
    const T *cur = mom[0];
    for (int e = 0; e < S.npath; ++e) {
        if (e > 0 && e % WAVE == 0) load_path(e);
        const int64_t slot = rl_l(p_slot, e % WAVE);
        T v = dot_row(Mr, cur);
        if (h != rl_i(p_half, e % WAVE)) v = T(0);
        v += __shfl_xor(v, 32);
        T *nx = L_.pv[q][e & 1];
        if (h == 0 && m < RMAX) nx[m] = v;
        if (slot >= 0 && h == 0 && m < r) partial[(slot * nq + q) * r + m] = v;
        wave_sync();
        cur = nx;
    }
    subtree_w<RMAX>(
        mats, del, mom, L_.dw[q], r, S.nnode, lane,
        [&](int n) {
            do ++n;
            while (n < S.nnode && rl_i(nd.cl, n) < 0);
            return n;
        },
        [&](int n) { return rl_i(nd.cl, n); },
        [&](int cl, int k, T v) { w[((int64_t)cl * nq + q) * r + k] = v; });
}

template <class T>
__device__ __forceinline__ T nanT() {
    return sizeof(T) == 8 ? (T)__builtin_nan("") : (T)__builtin_nanf("");
}

// Translation: one wavefront per cluster of the output side whose sources all
// lie in subtrees (a wavefront takes several in turn, the matrices in LDS);
// the clusters with a source above them ("heavy", first in the target list)
// take a workgroup, a source per wavefront. Lane (m, h) sums its row's half h
// of the columns l. A cluster has at most about four sources; their node
// values and nodes are staged four at a time in LDS with one round of loads.
// F formed from the nodes: eight or four terms of 1/d^m share a reciprocal as
// in the near field.
template <class T, int RMAX, int KB>
struct TrLds {
    alignas(16) T sw[WPB][4][KB][RMAX], st[WPB][4][RMAX];
    alignas(16) T zr[WPB][KB][RMAX];
    // A^T and D of the output side (before them A and D^T, for sources above the
    // subtrees); two matrices' rows in registers spilled
    T mat[RMAX * WAVE];
};
template <class T, int RMAX, bool TRANS, int SRC, int KID, int KB>
__device__ __forceinline__ void n1_translate_block(const DevPlanT<T> &p, const N1Side &o, int nq,
                                                   int blk, int nblk, const T *mats,
                                                   const T *partial, const T *w, T *z, int basis,
                                                   TrLds<T, RMAX, KB> &L_) {
    using Mt = N1Mat<T, RMAX>;
    constexpr bool FREE = SRC != N1_READ;
    constexpr int HALF = Mt::HALF, NB = 4, NT = HALF % 8 == 0 ? 8 : 4;
    auto &sw = L_.sw;
    auto &st = L_.st;
    auto &zr = L_.zr;
    const int lane = threadIdx.x % WAVE, wv = uniform((int)(threadIdx.x / WAVE));
    const int m = lane & 31, h = lane >> 5;
    const int r = p.r;
    const int mm = m < r ? m : 0;
    const T *oth = TRANS ? p.rnodes : p.cnodes;
    // a stored product: the source clusters with a basis value that is not finite
    // (a node meets a point), whose node values it makes NaN
    const uint8_t *bad = basis && p.odd[0] ? (TRANS ? p.bad_rc : p.bad_cc) : nullptr;
    const T *din = TRANS ? p.rdel : p.cdel, *dout = TRANS ? p.cdel : p.rdel;
    auto stage = [&](int from) {
#pragma unroll
        for (int e = 0; e < RMAX * WAVE; e += WG) L_.mat[e + threadIdx.x] = mats[from + e + threadIdx.x];
        __syncthreads();
    };
    T to = T(0), acc[KB];
#pragma unroll
    for (int k = 0; k < KB; ++k) acc[k] = T(0);
    // ws: zero past r (and past nq); ts: past r repeats
    auto apply = [&](const T (*ws)[RMAX], const T *ts, int64_t foff) {
        if constexpr (FREE && KB == 1) {
            const T acc0 = acc[0];
            const int l0 = h * HALF;
            bool odd = false;
#pragma unroll
            for (int j = 0; j < HALF; j += NT)
                odd |= near_terms<T, KID, TRANS, SRC == N1_EXACT, NT, 1>(
                    &to, ts + l0 + j, ws[0] + l0 + j, acc, 0, r - l0 - j);
            if constexpr (KID <= 2 && SRC == N1_FREE) {
                if (__builtin_expect(odd, 0)) {
                    T sum[1][1] = {{acc0}};
                    near_single<T, KID, TRANS, 1, 1>(&to, l0, min(l0 + HALF, r),
                                                     [&](int u, T &qu, T (&vu)[1]) {
                                                         qu = ts[u];
                                                         vu[0] = ws[0][u];
                                                     },
                                                     sum);
                    acc[0] = sum[0][0];
                }
            }
        } else {
            const T *F = p.F + foff;
            T fv[HALF];
#pragma unroll
            for (int j = 0; j < HALF; ++j) {
                if constexpr (FREE) {
                    const T t = ts[h * HALF + j];
                    fv[j] = TRANS ? kern_fast<T, KID>(t, to) : kern_fast<T, KID>(to, t);
                } else {
                    const int l = min(h * HALF + j, r - 1);
                    fv[j] = __builtin_nontemporal_load(TRANS ? F + (l + r * mm) : F + (mm + r * l));
                }
            }
#pragma unroll
            for (int j = 0; j < HALF; ++j)
#pragma unroll
                for (int k = 0; k < KB; ++k)
                    acc[k] = fmaT(h * HALF + j < r ? fv[j] : T(0), ws[k][h * HALF + j], acc[k]);
        }
    };
    auto put_z = [&] {  // this wavefront's sums into its zr
#pragma unroll
        for (int k = 0; k < KB; ++k) {
            acc[k] += __shfl_xor(acc[k], 32);
            if (h == 0 && m < RMAX) zr[wv][k][m] = m < r ? acc[k] : T(0);
            acc[k] = T(0);
        }
    };
    // c = A^T (z - d (D z)), d the lane's node offset; z: zs
    auto finish = [&](int id, T d, T (*zs)[RMAX]) {
        T c[KB];
        auto times = [&](const T *rows) {  // by one of the staged matrices, all z's together
#pragma unroll
            for (int k = 0; k < KB; ++k) c[k] = T(0);
#pragma unroll
            for (int j = 0; j < HALF; ++j) {
                const T a = rows[j * WAVE + lane];
#pragma unroll
                for (int k = 0; k < KB; ++k) c[k] = fmaT(a, zs[k][h * HALF + j], c[k]);
            }
#pragma unroll
            for (int k = 0; k < KB; ++k) c[k] += __shfl_xor(c[k], 32);
        };
        times(L_.mat + HALF * WAVE);
        wave_sync();
        if (h == 0 && m < RMAX) {
#pragma unroll
            for (int k = 0; k < KB; ++k) zs[k][m] -= d * c[k];
        }
        wave_sync();
        times(L_.mat);
        if (h == 0 && m < r) {
#pragma unroll
            for (int k = 0; k < KB; ++k)
                if (k < nq) z[((int64_t)id * nq + k) * r + m] = c[k];
        }
    };
    if (blk >= o.nheavy) {
        stage(Mt::AT);
        const int step = (nblk - o.nheavy) * WPB;
        for (int idx = o.nheavy + (blk - o.nheavy) * WPB + wv; idx < o.ncl; idx += step) {
            const N1Target C = sload_struct(o.target + idx);
            const T d = m < r ? dout[(int64_t)C.id * r + m] : T(0);
            if constexpr (FREE) to = (TRANS ? p.cnodes : p.rnodes)[(int64_t)C.id * r + mm];
            for (int e0 = C.beg; e0 < C.end; e0 += NB) {
                const int ne = min(NB, C.end - e0);
                // (source, right-hand side, column) = (i / KB RMAX, i / RMAX % KB, i % RMAX)
#pragma unroll
                for (int u = 0; u < (NB * KB * RMAX + WAVE - 1) / WAVE; ++u) {
                    const int i = lane + u * WAVE;
                    const int e = i / (KB * RMAX), k = i / RMAX % KB, l = i % RMAX;
                    if (e < ne) {
                        const int64_t src = o.tr[e0 + e].src;
                        T wl = w[(src * nq + min(k, nq - 1)) * r + min(l, r - 1)];
                        if (bad && bad[src]) wl = nanT<T>();
                        sw[wv][e][k][l] = l < r && k < nq ? wl : T(0);
                        if (FREE && k == 0) st[wv][e][l] = oth[src * r + min(l, r - 1)];
                    }
                }
                wave_sync();
#pragma unroll 1
                for (int e = 0; e < ne; ++e) apply(sw[wv][e], st[wv][e], FREE ? 0 : o.tr[e0 + e].foff);
                wave_sync();
            }
            put_z();
            wave_sync();
            finish(C.id, d, zr[wv]);
            wave_sync();
        }
        return;
    }
    stage(Mt::AU);
    const N1Target C = sload_struct(o.target + blk);
    if constexpr (FREE) to = (TRANS ? p.cnodes : p.rnodes)[(int64_t)C.id * r + mm];
    for (int e = C.beg + wv; e < C.end; e += WPB) {
        const DTrRec R = o.tr[e];
        if (FREE && h == 0 && m < RMAX) st[wv][0][m] = oth[(int64_t)R.src * r + (m < r ? m : r - 1)];
#pragma unroll 1
        for (int k = 0; k < KB; ++k) {
            const int kc = min(k, nq - 1);
            T wl;
            if (R.nslots > 0) {
                // lane half h sums the slots h, h + 2, ..., eight loads in flight
                // at 32-bit offsets (sixteen at 64-bit ones spilled)
                const T *ps = partial + (R.pbase * nq + kc) * r;
                const unsigned ld = 2u * nq * r;
                unsigned at = (unsigned)h * nq * r + mm;
                T s = T(0);
                int t = h;
                for (; t + 14 < R.nslots; t += 16, at += 8 * ld) {
                    T v[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) v[u] = ps[at + u * ld];
#pragma unroll
                    for (int u = 0; u < 8; ++u) s += v[u];
                }
                for (; t < R.nslots; t += 2, at += ld) s += ps[at];
                s += __shfl_xor(s, 32);
                if (h == 0 && m < RMAX) sw[wv][0][k][m] = m < r ? s : T(0);
                wave_sync();
                const T *mu[1] = {sw[wv][0][k]};
                const T d[1] = {m < r ? din[(int64_t)R.src * r + m] : T(0)};
                T v[1];
                node_values<RMAX, 1>(
                    [&](const T *u) { return dot_lds<T, HALF>(L_.mat, lane, u); },
                    [&](const T *u) { return dot_lds<T, HALF>(L_.mat + HALF * WAVE, lane, u); }, mu,
                    d, m, h, &zr[wv][k], v);
                wl = v[0];
            } else {
                wl = w[((int64_t)R.src * nq + kc) * r + mm];
            }
            if (bad && bad[R.src]) wl = nanT<T>();
            if (h == 0 && m < RMAX) sw[wv][0][k][m] = m < r && k < nq ? wl : T(0);
        }
        wave_sync();
        apply(sw[wv][0], st[wv][0], R.foff);
        wave_sync();
    }
    put_z();
    __syncthreads();
    stage(Mt::AT);
    if (wv != 0) return;
    for (int k = 0; k < KB; ++k) {
        T s = T(0);
        if (m < RMAX)
            for (int u = 0; u < WPB; ++u) s += zr[u][k][m];
        wave_sync();
        if (h == 0 && m < RMAX) zr[0][k][m] = s;
        wave_sync();
    }
    finish(C.id, m < r ? dout[(int64_t)C.id * r + m] : T(0), zr[0]);
}

// The two launches of the far-field chain before the downward pass. Each also
// takes about half of the near field's workgroups: the chain's are few and wait on
// latencies, and the near field does not depend on them.
//
// The two kinds alternate in groups of 256 workgroups, one for each CU, the
// chain's groups spread evenly among the near field's: with all of the chain's
// first they filled the chip alone (n = 2^20: 63 us), and alternating one by
// one or by eights, each kind met only half of the XCDs or of their shader
// engines, over which consecutive workgroups are dealt (84 us). Group g is the
// chain's number c(g) = floor(g n / total) if c(g + 1) > c(g), else the near
// field's number g - c(g); numbers past a kind's count do nothing.
constexpr int N1_GROUP = 256;
inline int n1_grid(int chain, int near) {
    return N1_GROUP * ((chain + N1_GROUP - 1) / N1_GROUP + (near + N1_GROUP - 1) / N1_GROUP);
}
__device__ __forceinline__ bool chain_block(int n, int &at) {
    const int g = (int)blockIdx.x / N1_GROUP, total = (int)gridDim.x / N1_GROUP;
    const int ng = (n + N1_GROUP - 1) / N1_GROUP;
    const int c0 = g * ng / total, c1 = (g + 1) * ng / total;
    at = N1_GROUP * (c1 > c0 ? c0 : g - c0) + (int)blockIdx.x % N1_GROUP;
    return c1 > c0;
}

// Five wavefronts per SIMD are asked of the register allocator where the near
// field is formed: left alone it gives four (upward) and three (translation);
// six cost the near field's chains their registers (85 us).
// Several right-hand sides: four, or three where the upward pass's LDS allows
// no more. Float32 up to rank 16: eight, which its registers allow (left alone,
// the scalar registers give seven: n = 500009, rank 10: 22.4 -> 24.4 us upward).
constexpr int n1_waves(int size, int src, int kid, int rmax, int kb) {
    if (size == 4 && rmax <= 16 && kid <= 2 && src != N1_READ && kb == 1) return 8;
    if (kid == 3 || (src == N1_READ && kb == 1)) return 1;
    return kb == 1 ? 5 : rmax > 24 || src == N1_READ ? 3 : 4;
}

template <class T, int RMAX, int SRC, int KID, bool TR, int KB>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(n1_waves(sizeof(T), SRC, KID, RMAX, KB))))
void k_n1_up(N1Side in, N1Side out, const T *in_pts, const T *out_pts, const T *A,
             const int32_t *odd, const T *mats, const T *del, MvArgsT<T> a, int r, int nq, int nup,
             int nb0, int nb) {
    __shared__ union Lds {
        std::conditional_t<KB == 1, UpLds<T, RMAX>, UpLdsKb<T, RMAX>> up;
        NearLds<T, KB> near;
        __device__ Lds() {}
    } s;
    int at;
    if (chain_block(nup, at)) {
        if (at >= nup) return;
        if constexpr (KB == 1)
            n1_up_block<T, RMAX>(in, in_pts, a.x, a.incx, mats, del, a.partial, a.w, r, at, s.up);
        else
            n1_up_block_kb<T, RMAX>(in, in_pts, a.x, a.incx, a.ldx, mats, del, a.partial, a.w, r, nq,
                                    at, s.up);
    } else if (at < nb) {
        near_block<T, KID, TR, SRC, KB>(out, at + nb0, out_pts, in_pts, A, odd, a, nq, s.near);
    }
}

template <class T, int RMAX, int SRC, int KID, bool TR, int KB>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(n1_waves(sizeof(T), SRC, KID, RMAX, KB))))
void k_n1_translate(DevPlanT<T> p, N1Side out, const T *in_pts, const T *out_pts, MvArgsT<T> a,
                    int nq, int ntr, int nb0, int nb) {
    __shared__ union Lds {
        TrLds<T, RMAX, KB> tr;
        NearLds<T, KB> near;
        __device__ Lds() {}
    } s;
    int at;
    if (chain_block(ntr, at)) {
        if (at < ntr)
            n1_translate_block<T, RMAX, TR, SRC, KID, KB>(p, out, nq, at, ntr, p.n1m, a.partial,
                                                          a.w, a.z, a.basis, s.tr);
    } else if (at < nb) {
        near_block<T, KID, TR, SRC, KB>(out, at + nb0, out_pts, in_pts, p.A, p.odd, a, nq,
                                        s.near);
    }
}

// The coefficients of a subtree's nodes into cof (LDS): the path's, one node
// after another, then each node's halves together (lane half h takes half h).
// z: ldz apart from cluster to cluster. One wavefront; pz: its LDS, sixteen path
// nodes' z at a time (and the last batch's final node in row N1_PATH); lane l
// holds local node l's record.
template <class T, int RMAX>
__device__ __forceinline__ void n1_coefficients(const N1Side &s, const N1Sub &S, const T *mats,
                                                const T *z, int64_t ldz, int r, int lane,
                                                T (*cof)[RMAX], T (*pz)[RMAX]) {
    using Mt = N1Mat<T, RMAX>;
    const int m = lane & 31, h = lane >> 5;
    N1Node nd{-1, {-1, -1}};
    N1Path P{-1, -1, 0};
    if (lane < S.nnode) nd = s.node[S.node + lane];
    if (lane < min(N1_PATH, S.npath)) P = s.path[S.path + lane];
    T Mr[RMAX];
    load_rows(mats + Mt::MD, lane, Mr);
    // the nodes' own z
    for (int i0 = 0; i0 < S.nnode * RMAX; i0 += WAVE) {
        const int i = i0 + lane, n = i / RMAX, l = i - n * RMAX;
        const int cl = __shfl(nd.cl, n < S.nnode ? n : 0);
        if (n < S.nnode) cof[n][l] = (cl >= 0 && l < r) ? z[cl * ldz + l] : T(0);
    }
    int half = 0;
    const T *cur = nullptr;
    for (int e0 = 0; e0 < S.npath; e0 += N1_PATH) {
        const int ne = min(N1_PATH, S.npath - e0);
        if (cur) {
            if (lane < ne) P = s.path[S.path + e0 + lane];
            wave_sync();
            if (h == 0 && m < RMAX) pz[N1_PATH][m] = cur[m];
            cur = pz[N1_PATH];
            wave_sync();
        }
#pragma unroll
        for (int u = 0; u < N1_PATH * RMAX / WAVE; ++u) {
            const int i = lane + u * WAVE, e = i / RMAX, l = i - e * RMAX;
            const int cl = __shfl(P.cl, e);
            if (e < ne) pz[e][l] = (cl >= 0 && l < r) ? z[cl * ldz + l] : T(0);
        }
        wave_sync();
        for (int e = 0; e < ne; ++e) {
            if (cur) {
                T v = dot_row(Mr, cur);
                if (h != half) v = T(0);
                v += __shfl_xor(v, 32);
                if (h == 0 && m < RMAX) pz[e][m] += v;
                wave_sync();
            }
            cur = pz[e];
            half = rl_i(P.half, e);
        }
    }
    wave_sync();
    if (cur) {
        T v = dot_row(Mr, cur);
        if (h != half) v = T(0);
        v += __shfl_xor(v, 32);
        if (h == 0 && m < RMAX) cof[0][m] += v;
        wave_sync();
    }
    for (int n = 0; n < S.nnode; ++n) {
        const int ca = rl_i(nd.c[0], n), cb = rl_i(nd.c[1], n);
        if (ca < 0 && cb < 0) continue;  // a leaf (wave-uniform)
        const int c = h ? cb : ca;
        const T v = dot_row(Mr, cof[n]);
        if (c >= 0 && m < RMAX) cof[c][m] += v;
        wave_sync();
    }
}

// One row of a chunk: the leaf's series by Clenshaw (coefficients in LDS, zero
// past r)
template <class T, int RMAX>
__device__ __forceinline__ T n1_series(const N1Chunk &C, const T (*cof)[RMAX], T p) {
    const T xh = ((p - (T)C.f.cx) - (T)C.f.cl) * (T)C.f.cy, x2 = xh + xh;
    const T *ck = cof[C.leaf];
    T b1 = T(0), b2 = T(0);
#pragma unroll
    for (int k = RMAX - 1; k >= 1; --k) {
        const T b0 = fmaT(x2, b1, ck[k] - b2);
        b2 = b1;
        b1 = b0;
    }
    return fmaT(xh, b1, ck[0] - b2);
}

// Downward pass: the far field added onto y, which holds the near field. A
// subtree per workgroup, its chunks over the wavefronts.
// Several right-hand sides: a wavefront forms the coefficients of each.
template <class T, int RMAX, int KB>
__global__ __launch_bounds__(WG) void k_n1_down(N1Side o, const T *pts_out, const T *z,
                                                const T *mats, const int32_t *odd,
                                                const uint8_t *bad_pt, MvArgsT<T> a, int r,
                                                int nq) {
    static_assert(KB <= WPB, "a wavefront per right-hand side");
    __shared__ __align__(16) T cof[KB][N1_NODES][RMAX];
    __shared__ __align__(16) T pz[KB][N1_PATH + 1][RMAX];
    const int lane = threadIdx.x % WAVE, wv = uniform((int)(threadIdx.x / WAVE));
    const N1Sub S = sload_struct(o.sub + blockIdx.x);
    // a stored product: the points with a basis value that is not finite, whose
    // rows it makes NaN
    const uint8_t *bad = a.basis && odd[0] ? bad_pt : nullptr;
    if (wv < nq)
        n1_coefficients<T, RMAX>(o, S, mats, z + wv * r, (int64_t)nq * r, r, lane, cof[wv], pz[wv]);
    __syncthreads();
    for (int c = S.ch + wv; c < S.ch + S.nch; c += WPB) {
        const N1Chunk C = sload_struct(o.ch + c);
        const int64_t at = C.p0 + min(lane, C.np - 1);
        const T po = pts_out[at];
        const bool nan = bad && bad[at];
#pragma unroll
        for (int k = 0; k < KB; ++k)
            if (k < nq) {
                const T v = n1_series<T, RMAX>(C, cof[k], po);
                n1_write(C, a, k, 1, lane, nan ? nanT<T>() : v);
            }
    }
}

// workgroups of the translation; light clusters: at most four wavefronts per
// SIMD, looping
inline int n1_ntranslate(const N1Side &out) {
    return out.nheavy + std::min((out.ncl - out.nheavy + WPB - 1) / WPB, 1024);
}

// the two launches without the near field (its workgroups: none)
template <class T, int RMAX, int KID, bool TR>
void n1_chain(const DevPlanT<T> &p, const MvArgsT<T> &a, hipStream_t s) {
    const N1Side &in = TR ? p.n1x : p.n1y, &out = TR ? p.n1y : p.n1x;
    const T *in_pts = TR ? p.x : p.y, *out_pts = TR ? p.y : p.x;
    const int ntr = n1_ntranslate(out);
    k_n1_up<T, RMAX, N1_FREE, KID, TR, 1><<<n1_grid(in.nsub, 0), WG, 0, s>>>(
        in, out, in_pts, out_pts, p.A, nullptr, p.n1m, TR ? p.rdel : p.cdel, a, p.r, 1, in.nsub, 0, 0);
    k_n1_translate<T, RMAX, N1_FREE, KID, TR, 1><<<n1_grid(ntr, 0), WG, 0, s>>>(
        p, out, in_pts, out_pts, a, 1, ntr, 0, 0);
}

// One product y = beta*y + op(H) x of nq <= KB right-hand sides over the
// interval trees. Many chunks of stored entries stream through k_down's near part,
// on the side stream when there is one.
template <class T, int RMAX, int SRC, int KID, bool TR, int KB>
hipError_t matvec_n1_t(const DevPlanT<T> &p, const MvArgsT<T> &a, int nq, hipStream_t s,
                       const hipEvent_t *ev) {
    auto mark = [&](int q) {
        if (ev) (void)hipEventRecord(ev[q], s);
    };
    const N1Side &in = TR ? p.n1x : p.n1y, &out = TR ? p.n1y : p.n1x;
    const T *in_pts = TR ? p.x : p.y, *out_pts = TR ? p.y : p.x;
    const bool far = p.nfar > 0;
    const bool stream = SRC == N1_READ && out.nunit > 0;
    const bool split = stream && a.side && !ev;
    auto near_part = [&](hipStream_t ns) {
        MvArgsT<T> an = a;
        an.part = 1;
        for (int q = 0; q < nq;) {
            an.y = a.y + q * a.ldy;
            an.x = a.x + q * a.ldx;
            if constexpr (TR) {
                k_down<T, RMAX, false, 0, true, true, 1><<<nblk(p.ncch), WG, 0, ns>>>(
                    p, p.cch, p.ncch, p.cnear, p.cfar, p.ccl, p.V, p.cmap, p.y, p.x, a.z, an);
                q += 1;
            } else if (nq - q == 4) {
                k_down<T, RMAX, false, 0, false, true, 4><<<nblk(p.nrch), WG, 0, ns>>>(
                    p, p.rch, p.nrch, p.rnear, p.rfar, p.rcl, p.U, p.rmap, p.x, p.y, a.z, an);
                q += 4;
            } else if (nq - q >= 2) {
                k_down<T, RMAX, false, 0, false, true, 2><<<nblk(p.nrch), WG, 0, ns>>>(
                    p, p.rch, p.nrch, p.rnear, p.rfar, p.rcl, p.U, p.rmap, p.x, p.y, a.z, an);
                q += 2;
            } else {
                k_down<T, RMAX, false, 0, false, true, 1><<<nblk(p.nrch), WG, 0, ns>>>(
                    p, p.rch, p.nrch, p.rnear, p.rfar, p.rcl, p.U, p.rmap, p.x, p.y, a.z, an);
                q += 1;
            }
        }
    };
    if (split) {
        hipError_t e = hipEventRecord(a.fork, s);
        if (e == hipSuccess) e = hipStreamWaitEvent(a.side, a.fork, 0);
        if (e != hipSuccess) return e;
        near_part(a.side);
        e = hipEventRecord(a.join, a.side);
        if (e != hipSuccess) return e;
    }
    // the near field's workgroups, five ninths with the upward pass, whose own
    // work is the smaller (n = 2^20: 68 and 67 us at one half each)
    const int nb = stream ? 0 : out.nunit > 0 ? (out.nunit + WPB - 1) / WPB : out.nch;
    const int nb0 = far ? (5 * nb + 8) / 9 : nb;
    const int nup = far ? in.nsub : 0;
    mark(0);
    if (nup + nb0 > 0)
        k_n1_up<T, RMAX, SRC, KID, TR, KB><<<n1_grid(nup, nb0), WG, 0, s>>>(
            in, out, in_pts, out_pts, p.A, p.odd, p.n1m, TR ? p.rdel : p.cdel, a, p.r, nq, nup, 0, nb0);
    mark(1);
    mark(2);
    if (far) {
        const int ntr = n1_ntranslate(out);
        k_n1_translate<T, RMAX, SRC, KID, TR, KB><<<n1_grid(ntr, nb - nb0), WG, 0, s>>>(
            p, out, in_pts, out_pts, a, nq, ntr, nb0, nb - nb0);
    }
    mark(3);
    if (split) {
        const hipError_t e = hipStreamWaitEvent(s, a.join, 0);
        if (e != hipSuccess) return e;
    } else if (stream) {
        near_part(s);
    }
    if (far)
        k_n1_down<T, RMAX, KB><<<out.nsub, WG, 0, s>>>(out, out_pts, a.z, p.n1m, p.odd,
                                                       TR ? p.bad_y : p.bad_x, a, p.r, nq);
    mark(4);
    return hipGetLastError();
}

// src: N1_FREE, N1_EXACT (kernels 1/d^m) or N1_READ
template <class T, int RMAX, bool TR, int KB>
hipError_t matvec_n1_k(const DevPlanT<T> &p, const MvArgsT<T> &a, int src, int nq, hipStream_t s,
                       const hipEvent_t *ev) {
    if (src == N1_READ) return matvec_n1_t<T, RMAX, N1_READ, 0, TR, KB>(p, a, nq, s, ev);
    // several right-hand sides form term by term either way
    if (src == N1_EXACT || (KB > 1 && p.kid <= 2)) {
        switch (p.kid) {
        case 0: return matvec_n1_t<T, RMAX, N1_EXACT, 0, TR, KB>(p, a, nq, s, ev);
        case 1: return matvec_n1_t<T, RMAX, N1_EXACT, 1, TR, KB>(p, a, nq, s, ev);
        default: return matvec_n1_t<T, RMAX, N1_EXACT, 2, TR, KB>(p, a, nq, s, ev);
        }
    }
    if constexpr (KB == 1) {
        switch (p.kid) {
        case 0: return matvec_n1_t<T, RMAX, N1_FREE, 0, TR, KB>(p, a, nq, s, ev);
        case 1: return matvec_n1_t<T, RMAX, N1_FREE, 1, TR, KB>(p, a, nq, s, ev);
        case 2: return matvec_n1_t<T, RMAX, N1_FREE, 2, TR, KB>(p, a, nq, s, ev);
        default: break;
        }
    }
    return matvec_n1_t<T, RMAX, N1_FREE, 3, TR, KB>(p, a, nq, s, ev);
}

template <class T, int RMAX>
hipError_t matvec_n1(const DevPlanT<T> &p, const MvArgsT<T> &a, bool tr, int src, int nq,
                     hipStream_t s, const hipEvent_t *ev) {
    if (nq == 1)
        return tr ? matvec_n1_k<T, RMAX, true, 1>(p, a, src, 1, s, ev)
                  : matvec_n1_k<T, RMAX, false, 1>(p, a, src, 1, s, ev);
    return tr ? matvec_n1_k<T, RMAX, true, N1_KB>(p, a, src, nq, s, ev)
              : matvec_n1_k<T, RMAX, false, N1_KB>(p, a, src, nq, s, ev);
}

}  // namespace
}  // namespace hmxk
