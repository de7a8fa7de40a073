// even.hip -- gfx950 kernels of the EvenBarycentricMatrix leaves
// (src/BarycentricMatrix.jl:5-89, mul! src/algebra.jl:168-239).
//
// Every pass is bound by HBM bandwidth: a product reads F (p x n) and W
// (n x m) once per leaf and does 2 flops per 8-byte factor entry.
#include "hmx_even.h"

namespace {

constexpr int WG = 256;

// W[k, i] = lambda_k * inv((2i-a-b-(b-a)x_k) * w_i), w_i = sum_k lambda_k *
// inv(2i-a-b-(b-a)x_k), src/BarycentricMatrix.jl:23-37 (and :62-75 for the
// m x n layout of barycentricmatrix), in the reference's operation order.
template <class T>
__global__ __launch_bounds__(WG) void k_even_gen_w(const ELeaf *leaves, int64_t nleaves,
                                                   ENodes<T> nd, int n, int layout, T *W, T *w) {
#pragma clang fp contract(off)
    for (int64_t t = blockIdx.y; t < nleaves; t += gridDim.y) {
        const ELeaf L = leaves[t];
        const T ba = (T)(L.b - L.a);
        for (int64_t i = (int64_t)blockIdx.x * WG + threadIdx.x; i < L.m;
             i += (int64_t)gridDim.x * WG) {
            const T c0 = (T)(2 * (L.a + i) - L.a - L.b);
            T s = T(0);
            for (int k = 0; k < n; ++k) s += nd.lam[k] * (T(1) / (c0 - ba * nd.x[k]));
            if (w) w[L.row0 + i] = s;
            T *out = W + L.woff;
            for (int k = 0; k < n; ++k) {
                const T v = nd.lam[k] * (T(1) / ((c0 - ba * nd.x[k]) * s));
                if (layout == 0) out[k + (int64_t)n * i] = v;
                else if (layout == 1) out[i + L.m * k] = v;
                else out[even_tile(i, k, n)] = v;
            }
        }
    }
}

// column-major staging copy of F -> 64-row tiles
template <class T>
__global__ __launch_bounds__(WG) void k_even_tile_F(const ELeaf *leaves, int64_t nleaves, int n,
                                                    const T *stage, T *F) {
    for (int64_t t = blockIdx.y; t < nleaves; t += gridDim.y) {
        const ELeaf L = leaves[t];
        const int64_t cnt = L.p * n;
        for (int64_t e = (int64_t)blockIdx.x * WG + threadIdx.x; e < cnt;
             e += (int64_t)gridDim.x * WG) {
            const int64_t k = e / L.p, j = e - k * L.p;
            F[L.foff + even_tile(j, k, n)] = stage[L.soff + e];
        }
    }
}

// Exchanges between lanes without LDS. v_permlane32_swap / v_permlane16_swap
// exchange the halves (odd and even rows of sixteen lanes) of two registers.
template <bool ROW>
__device__ inline void swap32(unsigned &a, unsigned &b) {
    if constexpr (ROW) {
        const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
        a = r[0];
        b = r[1];
    } else {
        const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
        a = r[0];
        b = r[1];
    }
}
template <bool ROW, class T>
__device__ inline T halve_swap(T a, T b) {
    constexpr int W = sizeof(T) / 4;
    unsigned x[W], y[W];
    __builtin_memcpy(x, &a, sizeof(T));
    __builtin_memcpy(y, &b, sizeof(T));
#pragma unroll
    for (int w = 0; w < W; ++w) swap32<ROW>(x[w], y[w]);
    __builtin_memcpy(&a, x, sizeof(T));
    __builtin_memcpy(&b, y, sizeof(T));
    return a + b;
}
template <int CTRL, class T>
__device__ inline T dpp(T v) {
    constexpr int W = sizeof(T) / 4;
    int x[W];
    __builtin_memcpy(x, &v, sizeof(T));
#pragma unroll
    for (int w = 0; w < W; ++w) x[w] = __builtin_amdgcn_update_dpp(0, x[w], CTRL, 0xf, 0xf, true);
    __builtin_memcpy(&v, x, sizeof(T));
    return v;
}
template <int CTRL, class T>
__device__ inline T halve_dpp(T a, T b, bool up) {
    return (up ? b : a) + dpp<CTRL>(up ? a : b);
}

// CB (8, 16 or 32) sums over the 32 lanes of each parity. Each step halves the
// sums a lane keeps: halves of the wavefront, rows of sixteen lanes, then within
// a row a rotation by four lanes (each lane ends with two neighbouring groups of
// four), by eight, and the pairs of a group of four. Returns the sum `even_col`.
constexpr int DPP_ROR4 = 0x124, DPP_ROR8 = 0x128, DPP_XOR2 = 0x4E;  // 0x4E: quad_perm 2 3 0 1
template <int CB, class T>
__device__ inline T halve_sums(T (&a)[CB], int lane) {
#pragma unroll
    for (int u = 0; u < CB / 2; ++u) a[u] = halve_swap<false>(a[u], a[u + CB / 2]);
#pragma unroll
    for (int u = 0; u < CB / 4; ++u) a[u] = halve_swap<true>(a[u], a[u + CB / 4]);
#pragma unroll
    for (int u = 0; u < CB / 8; ++u) a[u] = halve_dpp<DPP_ROR4>(a[u], a[u + CB / 8], lane & 4);
    if constexpr (CB >= 16) {
#pragma unroll
        for (int u = 0; u < CB / 16; ++u)
            a[u] = halve_dpp<DPP_ROR8>(a[u], a[u + CB / 16], lane & 8);
    } else {
        a[0] += dpp<DPP_ROR8>(a[0]);
    }
    if constexpr (CB >= 32) a[0] = halve_dpp<DPP_XOR2>(a[0], a[1], lane & 2);
    else a[0] += dpp<DPP_XOR2>(a[0]);
    return a[0];
}
// which sum a lane ends with
template <int CB>
__device__ inline int even_col(int lane) {
    const int c = (lane >> 5 & 1) * 16 | (lane >> 4 & 1) * 8 | (lane >> 2 & 1) * 4 |
                  (lane >> 3 & 1) * 2 | (lane >> 1 & 1);
    return c / (32 / CB);
}

// Upward pass: one workgroup per task. Thread t takes the task's columns
// t, t + 256, ..., so a lane's columns share one global parity; a wavefront's
// lanes of equal parity are summed, then the four wavefronts in LDS. Output
// e = (q*2 + par)*n + k of the leaf's beta (single-task leaves) or of the task's
// partial slot. Bound by reading F: one wavefront per task left the chip with 512
// (n = 2^18, rank 20, eight levels: 83 us), four with 3072 (55 us, 6.1 TB/s).
template <class T, int RB, int KB>
__global__ __launch_bounds__(WG) void k_even_up(EvenDev<T> p, const T *v, int64_t joff,
                                               int64_t incv, int64_t ldv, int nq) {
    constexpr int CB = RB <= 8 ? 8 : RB <= 16 ? 16 : 32;
    __shared__ T part[WG / 64][2 * KB * RB];
    const EUp tk = p.up[blockIdx.x];
    const ELeaf L = p.leaves[tk.leaf];
    const int n = p.n;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const T *F = p.F + L.foff;
    const int64_t jg = joff + L.col0;  // global column of the leaf's column 0
    T acc[KB][RB];
#pragma unroll
    for (int q = 0; q < KB; ++q)
#pragma unroll
        for (int k = 0; k < RB; ++k) acc[q][k] = T(0);
    const int64_t jend = tk.j0 + tk.len;
    for (int64_t j = tk.j0 + tid; j < jend; j += WG) {
        // all loads of the column first, then the products: each load is
        // guarded by k < n, and a guard around load and use would wait on
        // every load in turn. F is read once per product: non-temporal
        // loads (W, shared by the leaves of one size, stays cached instead)
        T x[KB], f[RB];
#pragma unroll
        for (int q = 0; q < KB; ++q) x[q] = q < nq ? v[q * ldv + (jg + j) * incv] : T(0);
        const T *Fj = F + even_tile(j, 0, n);
#pragma unroll
        for (int k = 0; k < RB; ++k) f[k] = k < n ? __builtin_nontemporal_load(Fj + k * EVEN_TILE) : T(0);
#pragma unroll
        for (int k = 0; k < RB; ++k)
#pragma unroll
            for (int q = 0; q < KB; ++q) acc[q][k] += f[k] * x[q];
    }
    const int par = (int)((jg + tk.j0 + lane) & 1);
#pragma unroll
    for (int q = 0; q < KB; ++q)
#pragma unroll
        for (int kb = 0; kb < RB; kb += CB) {
            T a[CB];
#pragma unroll
            for (int k = 0; k < CB; ++k) a[k] = kb + k < RB ? acc[q][kb + k] : T(0);
            const T val = halve_sums<CB>(a, lane);
            const int kk = kb + even_col<CB>(lane);
            if (kk < n) part[wv][(q * 2 + par) * n + kk] = val;
        }
    __syncthreads();
    const int64_t stride = (int64_t)HM_EVEN_KB * 2 * n;
    T *out = tk.single ? p.beta + (int64_t)tk.leaf * stride : p.partial + tk.slot * stride;
    for (int e = tid; e < 2 * KB * n; e += WG) {
        T t = part[0][e];
#pragma unroll
        for (int w = 1; w < WG / 64; ++w) t += part[w][e];
        out[e] = t;
    }
}

// beta of a leaf with several tasks: the sum of its partials; thread
// (g, e) sums slots g, g + G, ... of entry e, then the G partial sums are
// added in g order. With more than 256 entries (2 parities x kb right-hand
// sides x rank n) each thread sums whole entries e, e + 256, ... in slot order.
template <class T>
__global__ __launch_bounds__(256) void k_even_reduce(EvenDev<T> p, int kb) {
    const ERed r = p.red[blockIdx.x];
    const int64_t stride = (int64_t)HM_EVEN_KB * 2 * p.n;
    const int E = 2 * kb * p.n;
    if (E > 256) {  // block-uniform: no thread reaches the barrier below
        for (int e = threadIdx.x; e < E; e += 256) {
            T s = T(0);
            for (int t = 0; t < r.ntask; ++t) s += p.partial[(r.slot0 + t) * stride + e];
            p.beta[(int64_t)r.leaf * stride + e] = s;
        }
        return;
    }
    const int G = 256 / E;
    const int e = threadIdx.x % E, g = threadIdx.x / E;
    __shared__ T part[256];
    T s = T(0);
    if (g < G)
        // eight loads in flight; the sum keeps slot order
        for (int t = g; t < r.ntask; t += 8 * G) {
            T v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                v[u] = t + u * G < r.ntask ? p.partial[(r.slot0 + t + u * G) * stride + e] : T(0);
#pragma unroll
            for (int u = 0; u < 8; ++u) s += v[u];
        }
    part[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x < E) {
        T tot = T(0);
        for (int q = 0; q < G; ++q) tot += part[q * E + threadIdx.x];
        p.beta[(int64_t)r.leaf * stride + threadIdx.x] = tot;
    }
}

// Downward pass: one thread per row of a segment. Row I pairs with the
// columns of its own parity (I + J even), so it takes beta[I % 2]. W is in
// 64-row tiles, so a wavefront's loads of one k are one contiguous run; the
// current leaf's beta is staged in LDS (two distinct addresses per wave).
template <class T, int RB, int KB>
__global__ __launch_bounds__(WG) void k_even_down(EvenDev<T> p, T *u, int64_t ioff, int64_t incu,
                                                  int64_t ldu, int nq, int store) {
    __shared__ T sb[2 * KB * RB];
    const EDown d = p.down[blockIdx.x];
    const int tid = threadIdx.x;
    const bool valid = tid < d.len;
    const int n = p.n;
    const int64_t r = d.r0 + (valid ? tid : 0);
    const int par = (int)((ioff + r) & 1);
    const int64_t stride = (int64_t)HM_EVEN_KB * 2 * n;
    T s[KB];
#pragma unroll
    for (int q = 0; q < KB; ++q) s[q] = T(0);
    for (int e = d.lbeg; e < d.lend; ++e) {
        const int32_t id = p.list[e];
        const ELeaf L = p.leaves[id];
        __syncthreads();
        for (int t = tid; t < 2 * KB * n; t += WG) sb[t] = p.beta[(int64_t)id * stride + t];
        __syncthreads();
        if (valid) {
            const T *wr = p.W + L.woff + even_tile(r - L.row0, 0, n);
            T wk[RB];
#pragma unroll
            for (int k = 0; k < RB; ++k) wk[k] = k < n ? wr[k * EVEN_TILE] : T(0);
#pragma unroll
            for (int q = 0; q < KB; ++q) {
                const T *bq = sb + (q * 2 + par) * n;
                T a = T(0);
#pragma unroll
                for (int k = 0; k < RB; ++k)
                    if (k < n) a += wk[k] * bq[k];
                s[q] += a;
            }
        }
    }
    if (valid) {
#pragma unroll
        for (int q = 0; q < KB; ++q) {
            if (q < nq) {
                T *uo = u + q * ldu + (ioff + r) * incu;
                *uo = store ? s[q] : *uo + s[q];
            }
        }
    }
}

template <class T>
__global__ __launch_bounds__(WG) void k_even_zero(T *u, int64_t ioff, int64_t incu, int64_t ldu,
                                                  int64_t nrows, int nq) {
    const int64_t i = (int64_t)blockIdx.x * WG + threadIdx.x;
    if (i >= nrows) return;
    for (int q = 0; q < nq; ++q) u[q * ldu + (ioff + i) * incu] = T(0);
}

template <class T, int RB, int KB>
hipError_t even_matvec_t(const EvenDev<T> &p, T *u, const T *v, int64_t ioff, int64_t joff,
                         int64_t incu, int64_t incv, int64_t ldu, int64_t ldv, int nq, int beta,
                         hipStream_t s) {
    for (int q0 = 0; q0 < nq; q0 += KB) {
        const int nb = nq - q0 < KB ? nq - q0 : KB;
        T *uq = u + q0 * ldu;
        const T *vq = v + q0 * ldv;
        // beta = 0: rows of a segment are written by the downward pass;
        // rows no leaf covers are cleared first
        const int store = beta == 0 && p.covered;
        if (beta == 0 && !p.covered && p.nrows > 0)
            k_even_zero<T><<<(unsigned)((p.nrows + WG - 1) / WG), WG, 0, s>>>(uq, ioff, incu, ldu,
                                                                          p.nrows, nb);
        if (p.nup > 0) k_even_up<T, RB, KB><<<p.nup, WG, 0, s>>>(p, vq, joff, incv, ldv, nb);
        if (p.nred > 0) k_even_reduce<T><<<p.nred, 256, 0, s>>>(p, nb);
        if (p.ndown > 0) k_even_down<T, RB, KB><<<p.ndown, WG, 0, s>>>(p, uq, ioff, incu, ldu, nb,
                                                                  store);
    }
    return hipGetLastError();
}

template <class T>
hipError_t gen_weights_t(const ELeaf *leaves, int64_t nleaves, int64_t max_m, const ENodes<T> &nodes,
                         int n, int layout, T *W, T *w, hipStream_t s) {
    if (nleaves <= 0 || max_m <= 0) return hipSuccess;
    const int64_t bx = (max_m + WG - 1) / WG;
    dim3 grid((unsigned)(bx < 1024 ? bx : 1024), (unsigned)(nleaves < 65535 ? nleaves : 65535));
    k_even_gen_w<T><<<grid, WG, 0, s>>>(leaves, nleaves, nodes, n, layout, W, w);
    return hipGetLastError();
}

template <class T>
hipError_t tile_F_t(const ELeaf *leaves, int64_t nleaves, int64_t max_pn, int n, const T *stage,
                    T *F, hipStream_t s) {
    if (nleaves <= 0 || max_pn <= 0) return hipSuccess;
    const int64_t bx = (max_pn + WG - 1) / WG;
    dim3 grid((unsigned)(bx < 4096 ? bx : 4096), (unsigned)(nleaves < 65535 ? nleaves : 65535));
    k_even_tile_F<T><<<grid, WG, 0, s>>>(leaves, nleaves, n, stage, F);
    return hipGetLastError();
}

template <class T>
hipError_t matvec_dispatch(const EvenDev<T> &p, T *u, const T *v, int64_t ioff, int64_t joff,
                           int64_t incu, int64_t incv, int64_t ldu, int64_t ldv, int nq, int beta,
                           hipStream_t s) {
    const int n = p.n;
    if (nq == 1) {  // one right-hand side: the single-column kernels (fewer registers)
        if (n <= 8) return even_matvec_t<T, 8, 1>(p, u, v, ioff, joff, incu, incv, ldu, ldv, nq, beta, s);
        if (n <= 16) return even_matvec_t<T, 16, 1>(p, u, v, ioff, joff, incu, incv, ldu, ldv, nq, beta, s);
        if (n <= 24) return even_matvec_t<T, 24, 1>(p, u, v, ioff, joff, incu, incv, ldu, ldv, nq, beta, s);
        if (n <= 32) return even_matvec_t<T, 32, 1>(p, u, v, ioff, joff, incu, incv, ldu, ldv, nq, beta, s);
    }
    if (n <= 8) return even_matvec_t<T, 8, 4>(p, u, v, ioff, joff, incu, incv, ldu, ldv, nq, beta, s);
    if (n <= 16) return even_matvec_t<T, 16, 4>(p, u, v, ioff, joff, incu, incv, ldu, ldv, nq, beta, s);
    if (n <= 24) return even_matvec_t<T, 24, 2>(p, u, v, ioff, joff, incu, incv, ldu, ldv, nq, beta, s);
    if (n <= 32) return even_matvec_t<T, 32, 2>(p, u, v, ioff, joff, incu, incv, ldu, ldv, nq, beta, s);
    if (n <= 48) return even_matvec_t<T, 48, 1>(p, u, v, ioff, joff, incu, incv, ldu, ldv, nq, beta, s);
    return even_matvec_t<T, 64, 1>(p, u, v, ioff, joff, incu, incv, ldu, ldv, nq, beta, s);
}

}  // namespace

hipError_t hmx_even_gen_weights(const ELeaf *leaves, int64_t nleaves, int64_t max_m,
                                const ENodes<double> &nodes, int n, int layout, double *W,
                                double *w, hipStream_t s) {
    return gen_weights_t<double>(leaves, nleaves, max_m, nodes, n, layout, W, w, s);
}
hipError_t hmx_even_gen_weights(const ELeaf *leaves, int64_t nleaves, int64_t max_m,
                                const ENodes<float> &nodes, int n, int layout, float *W,
                                float *w, hipStream_t s) {
    return gen_weights_t<float>(leaves, nleaves, max_m, nodes, n, layout, W, w, s);
}

hipError_t hmx_even_tile_F(const ELeaf *leaves, int64_t nleaves, int64_t max_pn, int n,
                           const double *stage, double *F, hipStream_t s) {
    return tile_F_t<double>(leaves, nleaves, max_pn, n, stage, F, s);
}
hipError_t hmx_even_tile_F(const ELeaf *leaves, int64_t nleaves, int64_t max_pn, int n,
                           const float *stage, float *F, hipStream_t s) {
    return tile_F_t<float>(leaves, nleaves, max_pn, n, stage, F, s);
}

hipError_t hmx_even_matvec(const EvenDev<double> &p, double *u, const double *v, int64_t ioff,
                           int64_t joff, int64_t incu, int64_t incv, int64_t ldu, int64_t ldv,
                           int nq, int beta, hipStream_t s) {
    return matvec_dispatch<double>(p, u, v, ioff, joff, incu, incv, ldu, ldv, nq, beta, s);
}
hipError_t hmx_even_matvec(const EvenDev<float> &p, float *u, const float *v, int64_t ioff,
                           int64_t joff, int64_t incu, int64_t incv, int64_t ldu, int64_t ldv,
                           int nq, int beta, hipStream_t s) {
    return matvec_dispatch<float>(p, u, v, ioff, joff, incu, incv, ldu, ldv, nq, beta, s);
}
