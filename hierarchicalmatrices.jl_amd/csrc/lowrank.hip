// lowrank.hip -- gfx950 kernels of the batched LowRankMatrix arithmetic
// (src/LowRankMatrix.jl:64-171). One workgroup per item (and side) in every
// launch:
//   k_lr_pack    tall factors to factor: [U1 U2], [V1 V2], A or A^T
//   k_lr_gemm    tall x small products: A U2 and A^T V1 before the QR, and
//                U1 SU, V1 SU, V2 SV after the SVD
//   k_lr_gram    M = X1^T U2 (cores of L1 * L2 and L1' * L2)
//   k_lr_qr      Householder QR in place (LAPACK dlarfg convention: beta =
//                -sign(alpha) ||x||, tau = (beta - alpha)/beta, v(1) = 1) and T
//                of the compact WY form Q = I - V T V^T (LAPACK dlarft
//                recurrence over the Gram matrix V^T V)
//   k_lr_svd     core, one-sided Jacobi SVD in LDS, descending order, getrank
//   k_lr_wz      W = T (V^T [S_; 0]) for the compact WY product
//   k_lr_applyq  Q [S_; 0] = [S_; 0] - V W, one pass over V
#include "hmx.h"
#include "hmx_lowrank.h"

namespace {

constexpr int WG = 256;
constexpr int LD = LR_MAX + 1;  // LDS leading dimension of the Jacobi matrices

struct TallView {
    double *X;    // M x C, column-major, ld M
    int M, C;
    double *R;    // C x C (ld LR_MAX) in the small slot
    double *T;    // C x C compact-WY factor (ld LR_MAX)
    double *tau;  // C
};

__device__ inline TallView tall_view(const LRItem &it, int side, double *tall, double *small) {
    double *sl = small + it.small;
    TallView v;
    v.X = tall + (side ? it.xv : it.xu);
    v.M = side ? it.n : it.m;
    v.C = side ? it.cv : it.cu;
    v.R = sl + (side ? LR_RV : LR_RU);
    v.T = sl + (side ? LR_WV : LR_WU);
    v.tau = sl + (side ? LR_TV : LR_TU);
    return v;
}

// [U1 U2] -> XU, [V1 V2] -> XV (sums); A -> XU or A^T -> XV (svdtrunc)
__global__ __launch_bounds__(WG) void k_lr_pack(int op, const LRItem *items, double *tall) {
    const LRItem it = items[blockIdx.x];
    const int side = blockIdx.y;
    const int C = side ? it.cv : it.cu;
    if (C == 0) return;
    const int M = side ? it.n : it.m;
    double *X = tall + (side ? it.xv : it.xu);
    const int64_t cnt = (int64_t)M * C;
    for (int64_t e = (int64_t)blockIdx.z * WG + threadIdx.x; e < cnt; e += (int64_t)gridDim.z * WG) {
        const int i = (int)(e % M), c = (int)(e / M);
        double v;
        if (op == HM_LR_SVDTRUNC) {
            v = side ? it.A[c + (int64_t)it.m * i] : it.A[e];
        } else {
            const double *F1 = side ? it.V1 : it.U1, *F2 = side ? it.V2 : it.U2;
            v = c < it.r1 ? F1[i + (int64_t)M * c] : F2[i + (int64_t)M * (c - it.r1)];
        }
        X[e] = v;
    }
}

// out (rows x R, ld rows) = X (rows x P) B (P x R); X(i, t) = X[i*si + t*st]
// (X == nullptr: the identity), B(t, c) = B[t*b0 + c*b1]. B goes through
// LDS in chunks of 64 rows; one thread per output row.
struct GemmDesc {
    const double *X;
    int64_t si, st;
    const double *B;
    int64_t b0, b1;
    double *out;
    int rows, P, R;
};

__device__ inline bool gemm_desc(int op, const LRItem &it, int stage, int side, double *tall,
                                 double *small, GemmDesc &g) {
    const double *sl = small + it.small;
    g.X = nullptr;
    g.si = 1;
    g.st = 0;
    if (stage == 0) {  // before the QR: the tall factor of A * L or L * A
        if (op == HM_LR_DMUL && side == 0) {
            g.X = it.A; g.si = 1; g.st = it.m;
            g.B = it.U2; g.b0 = 1; g.b1 = it.k;
            g.out = tall + it.xu; g.rows = it.m; g.P = it.k; g.R = it.r2;
            return true;
        }
        if (op == HM_LR_MULD && side == 1) {
            g.X = it.A; g.si = it.k; g.st = 1;
            g.B = it.V1; g.b0 = 1; g.b1 = it.k;
            g.out = tall + it.xv; g.rows = it.n; g.P = it.k; g.R = it.r1;
            return true;
        }
        return false;
    }
    // after the SVD: sides without a QR factor
    if ((side ? it.cv : it.cu) != 0) return false;
    g.R = (int)sl[LR_RANK];
    g.B = sl + (side ? LR_SV : LR_SU);
    g.b0 = 1;
    g.b1 = LR_MAX;
    if (side == 0) {
        g.out = it.Uo; g.rows = it.m;
        if (op == HM_LR_MUL || op == HM_LR_MULD) { g.X = it.U1; g.st = it.m; g.P = it.r1; }
        else if (op == HM_LR_ADJMUL) { g.X = it.V1; g.st = it.m; g.P = it.r1; }
        else { g.X = nullptr; g.P = it.m; }  // svdtrunc of A^T: U = SU
    } else {
        g.out = it.Vo; g.rows = it.n;
        if (op == HM_LR_MUL || op == HM_LR_ADJMUL || op == HM_LR_DMUL) {
            g.X = it.V2; g.st = it.n; g.P = it.r2;
        } else { g.X = nullptr; g.P = it.n; }  // svdtrunc of A: V = SV
    }
    return true;
}

template <int RB>
__global__ __launch_bounds__(WG) void k_lr_gemm(int op, int stage, const LRItem *items,
                                                double *tall, double *small) {
    const LRItem it = items[blockIdx.x];
    GemmDesc g;
    if (!gemm_desc(op, it, stage, blockIdx.y, tall, small, g)) return;
    const int row0 = blockIdx.z * WG;
    if (row0 >= g.rows) return;
    const int i = row0 + threadIdx.x;
    const bool valid = i < g.rows;
    __shared__ double bs[64 * RB];
    double acc[RB];
#pragma unroll
    for (int c = 0; c < RB; ++c) acc[c] = 0.0;
    for (int t0 = 0; t0 < g.P; t0 += 64) {
        const int tl = min(64, g.P - t0);
        __syncthreads();
        for (int e = threadIdx.x; e < tl * g.R; e += WG) {
            const int t = e % tl, c = e / tl;
            bs[t + 64 * c] = g.B[(int64_t)(t0 + t) * g.b0 + (int64_t)c * g.b1];
        }
        __syncthreads();
        if (valid) {
            for (int t = 0; t < tl; ++t) {
                const double x = g.X ? g.X[(int64_t)i * g.si + (int64_t)(t0 + t) * g.st]
                                     : (i == t0 + t ? 1.0 : 0.0);
#pragma unroll
                for (int c = 0; c < RB; ++c)
                    if (c < g.R) acc[c] += x * bs[t + 64 * c];
            }
        }
    }
    if (valid) {
#pragma unroll
        for (int c = 0; c < RB; ++c)
            if (c < g.R) g.out[i + (int64_t)g.rows * c] = acc[c];
    }
}

// M (r1 x r2, ld LR_MAX, in the RU place) = X1^T U2 over k rows; X1 = V1
// (L1 * L2) or U1 (L1' * L2). Rows stream through LDS in chunks of 32.
__global__ __launch_bounds__(WG) void k_lr_gram(int op, const LRItem *items, double *small) {
    const LRItem it = items[blockIdx.x];
    const double *X1 = op == HM_LR_MUL ? it.V1 : it.U1;
    const double *X2 = it.U2;
    const int K = it.k, A = it.r1, B = it.r2;
    __shared__ double t1[32 * LR_MAX], t2[32 * LR_MAX];
    double acc[16];
#pragma unroll
    for (int o = 0; o < 16; ++o) acc[o] = 0.0;
    const int nout = A * B;
    for (int t0 = 0; t0 < K; t0 += 32) {
        const int tl = min(32, K - t0);
        for (int e = threadIdx.x; e < tl * A; e += WG) {
            const int t = e % tl, a = e / tl;
            t1[t + 32 * a] = X1[(int64_t)a * K + t0 + t];
        }
        for (int e = threadIdx.x; e < tl * B; e += WG) {
            const int t = e % tl, b = e / tl;
            t2[t + 32 * b] = X2[(int64_t)b * K + t0 + t];
        }
        __syncthreads();
#pragma unroll
        for (int o = 0; o < 16; ++o) {
            const int e = threadIdx.x + o * WG;
            if (e < nout) {
                const int a = e % A, b = e / A;
                double s = 0.0;
                for (int t = 0; t < tl; ++t) s += t1[t + 32 * a] * t2[t + 32 * b];
                acc[o] += s;
            }
        }
        __syncthreads();
    }
    double *M = small + it.small + LR_RU;
#pragma unroll
    for (int o = 0; o < 16; ++o) {
        const int e = threadIdx.x + o * WG;
        if (e < nout) M[(e % A) + LR_MAX * (e / A)] = acc[o];
    }
}

// Exchanges between lanes without LDS
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E;  // quad_perm 1 0 3 2, 2 3 0 1
constexpr int DPP_HALF_MIRROR = 0x141, DPP_MIRROR = 0x140, DPP_ROR8 = 0x128;
template <int CTRL>
__device__ inline double dpp(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// CB sums over the 64 lanes, one column per 64 / CB lanes: returns the sum of
// column lane / (64 / CB). Each step halves the columns a lane keeps: upper and
// lower half of the wavefront, rows of sixteen lanes (v_permlane32_swap,
// v_permlane16_swap: lane l's a + b is the sum for a where the exchanged bit
// of l is 0 and for b where it is 1), then DPP.
template <int CTRL>
__device__ inline double halve_dpp(double a, double b, bool up) {
    return (up ? b : a) + dpp<CTRL>(up ? a : b);
}
template <bool ROW>
__device__ inline double halve_swap(double a, double b) {
    const unsigned al = __double2loint(a), ah = __double2hiint(a), bl = __double2loint(b),
                   bh = __double2hiint(b);
    if constexpr (ROW) {
        const auto l = __builtin_amdgcn_permlane16_swap(al, bl, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap(ah, bh, false, false);
        return __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
    } else {
        const auto l = __builtin_amdgcn_permlane32_swap(al, bl, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap(ah, bh, false, false);
        return __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
    }
}
template <int CB>
__device__ inline double halve_sums(double (&a)[CB], int lane) {
#pragma unroll
    for (int u = 0; u < CB / 2; ++u) a[u] = halve_swap<false>(a[u], a[u + CB / 2]);
#pragma unroll
    for (int u = 0; u < CB / 4; ++u) a[u] = halve_swap<true>(a[u], a[u + CB / 4]);
#pragma unroll
    for (int u = 0; u < CB / 8; ++u) a[u] = halve_dpp<DPP_ROR8>(a[u], a[u + CB / 8], lane & 8);
    if constexpr (CB >= 16) {
#pragma unroll
        for (int u = 0; u < CB / 16; ++u)
            a[u] = halve_dpp<DPP_HALF_MIRROR>(a[u], a[u + CB / 16], lane & 4);
    } else {
        a[0] += dpp<DPP_HALF_MIRROR>(a[0]);
    }
    if constexpr (CB >= 32) {
#pragma unroll
        for (int u = 0; u < CB / 32; ++u)
            a[u] = halve_dpp<DPP_XOR2>(a[u], a[u + CB / 32], lane & 2);
    } else {
        a[0] += dpp<DPP_XOR2>(a[0]);
    }
    if constexpr (CB >= 64) a[0] = halve_dpp<DPP_XOR1>(a[0], a[1], lane & 1);
    else a[0] += dpp<DPP_XOR1>(a[0]);
    return a[0];
}

// Householder QR in place (LAPACK dlarfg convention: beta = -sign(alpha) *
// norm, tau = (beta - alpha) / beta, v = [1; x[j+1:] / (alpha - beta)]): the
// reflectors below X's diagonal, R (upper C x C, ld LR_MAX) and tau into the
// small slot. X's upper triangle is left as it falls: nothing reads it.
//
// Panels of PW = 8 columns, then the columns to their right eight at a time. One
// workgroup of 512 threads; thread t owns rows t, t + WGR, ... throughout, so the
// passes over X need no barrier between them, only the sums over rows do.
//
// qr_panel: the first RR rows of a thread stay in registers for the panel's
// steps, the rest are streamed. A row keeps its trailing columns only: x[q] is
// column j + q, and the update of step j writes x[q - 1]. One pass per step both
// updates the rows and forms the next step's dot products x_{j+1}[j+2:] .
// x_k[j+2:] (q = 0: the squared norm), so a step has one barrier: the sums are
// halved over the wavefront's lanes, then every wavefront adds the wavefronts'
// and forms beta, tau and w_k = tau (x_k[j] + v[j+1:] . x_k[j+1:]) for itself.
// The thread of row j + 1 leaves it in LDS instead of adding it to the sums.
//
// panel_sums and panel_update: S = V^T B for eight columns B (or the panel's own:
// its Gram matrix G), one sum a lane; the eight reflectors in turn are then
// w_j = tau_j (S_j - sum_{l<j} G_lj w_l), and B -= V w.
//
// Updating every trailing column in every step instead (rows in registers where
// they fit) streams the rest of X through L2 once a step, at one compute unit's
// 64 bytes a cycle: 295 us with T for differences of 20 blocks of 256 to 2048
// rows and 10 to 32 columns; in panels 181. Two passes per step, eight
// columns at a time, took 640 (779 with the factors held in LDS, a launch of its
// own) and T another 412.
constexpr int WGR = 512, NWR = WGR / 64, PW = 8;
constexpr int RR = 4;  // 2048 rows in registers (six or eight: spills)

struct QrLds {
    double red[2][NWR][PW], row[2][PW], sums[2][NWR][PW * PW];
};

__device__ inline double lane_value(double v, int lane) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
    return __hiloint2double(hi, lo);
}

// columns p0 .. p0 + C - 1 (C <= PW), rows p0 .. M - 1
__device__ inline void qr_panel(const TallView &T, int p0, int C, QrLds &s) {
    const int M = T.M;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    double *const X = T.X + (int64_t)p0 * M;
    double x[RR][PW], acc[PW];
#pragma unroll
    for (int q = 0; q < PW; ++q) acc[q] = 0.0;
#pragma unroll
    for (int k = 0; k < RR; ++k) {
        if (WGR * k >= M) break;
        const int i = tid + WGR * k;
#pragma unroll
        for (int q = 0; q < PW; ++q)
            x[k][q] = q < C && i >= p0 && i < M ? X[(int64_t)q * M + i] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < RR; ++k) {
        if (WGR * k >= M) break;
        const double x0 = tid + WGR * k > p0 ? x[k][0] : 0.0;
#pragma unroll
        for (int q = 0; q < PW; ++q) acc[q] += x0 * x[k][q];
    }
    if (tid == p0) {
#pragma unroll
        for (int q = 0; q < PW; ++q) s.row[0][q] = x[0][q];
    }
    for (int i0 = WGR * RR; i0 < M; i0 += WGR) {
        const int i = min(i0 + tid, M - 1);
        const double x0 = i0 + tid < M ? X[i] : 0.0;
#pragma unroll
        for (int q = 0; q < PW; ++q) acc[q] += x0 * X[(int64_t)min(q, C - 1) * M + i];
    }
    for (int jl = 0; jl < C; ++jl) {
        const int j = p0 + jl, nk = C - jl, b = jl & 1;
        const double wsum = halve_sums<PW>(acc, lane);
        if ((lane & 7) == 0) s.red[b][wv][lane >> 3] = wsum;
        __syncthreads();
        const int ql = lane & (PW - 1);
        double sum = 0.0;
#pragma unroll
        for (int w = 0; w < NWR; ++w) sum += s.red[b][w][ql];
        const double rj = s.row[b][ql];
        const double xn2 = lane_value(sum, 0), alpha = lane_value(rj, 0);
        double beta = alpha, t = 0.0, scal = 1.0;
        if (xn2 > 0.0) {
            beta = -copysign(sqrt(alpha * alpha + xn2), alpha);
            t = (beta - alpha) / beta;
            scal = 1.0 / (alpha - beta);
        }
        const double wl = t != 0.0 && ql < nk ? t * (rj + scal * sum) : 0.0;
        if (wv == 0 && lane < nk) {
            T.R[j + LR_MAX * (j + lane)] = lane == 0 ? beta : rj - wl;
            if (lane == 0) T.tau[j] = t;
        }
        double w[PW];
#pragma unroll
        for (int q = 1; q < PW; ++q) w[q] = lane_value(wl, q);
#pragma unroll
        for (int q = 0; q < PW; ++q) acc[q] = 0.0;
#pragma unroll
        for (int k = 0; k < RR; ++k) {
            // rows up to j and past M go along unstored (a branch would keep
            // two copies of the row in registers)
            if (WGR * k >= M) break;
            const int i = tid + WGR * k;
            const double v = x[k][0] * scal;
            if (i > j && i < M) X[(int64_t)jl * M + i] = v;
            const double vv = t != 0.0 && i > j ? v : 0.0;
#pragma unroll
            for (int q = 1; q < PW; ++q) x[k][q - 1] = x[k][q] - w[q] * vv;
            x[k][PW - 1] = 0.0;
            const double x0 = i > j + 1 ? x[k][0] : 0.0;
#pragma unroll
            for (int q = 0; q < PW; ++q) acc[q] += x0 * x[k][q];
        }
        if (tid == j + 1) {
#pragma unroll
            for (int q = 0; q < PW; ++q) s.row[b ^ 1][q] = x[0][q];
        }
        for (int i0 = WGR * RR; i0 < M; i0 += WGR) {
            // columns past the last are read as the last and not stored
            const int i = min(i0 + tid, M - 1);
            const bool own = i0 + tid < M;
            double *xr = X + (int64_t)jl * M + i;
            double y[PW];
#pragma unroll
            for (int q = 0; q < PW; ++q) y[q] = xr[(int64_t)min(q, nk - 1) * M];
            const double v = y[0] * scal, vv = t != 0.0 ? v : 0.0;
            if (own) xr[0] = v;
#pragma unroll
            for (int q = 1; q < PW; ++q) {
                y[q] -= w[q] * vv;
                if (own && q < nk) xr[(int64_t)q * M] = y[q];
            }
            const double x0 = own && nk > 1 ? y[1] : 0.0;
#pragma unroll
            for (int q = 1; q < PW; ++q) acc[q - 1] += x0 * y[q];
        }
    }
}

// V^T B over the rows: lane 8 a + c receives v_a . B_c, for the panel's V (unit
// lower triangular from row p0) and B = columns c0 .. of X (cn of them; those
// past the last count as the last), or V itself (c0 == p0)
__device__ inline double panel_sums(const TallView &T, int p0, int c0, int cn, QrLds &s, int b) {
    const int M = T.M, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const double *V = T.X + (int64_t)p0 * M, *B = T.X + (int64_t)c0 * M;
    double acc[PW * PW];
#pragma unroll
    for (int e = 0; e < PW * PW; ++e) acc[e] = 0.0;
    for (int i0 = 0; i0 < M; i0 += WGR) {
        const int i = min(i0 + tid, M - 1);
        const bool own = i0 + tid < M && i >= p0;
        double v[PW], x[PW];
#pragma unroll
        for (int a = 0; a < PW; ++a) v[a] = V[(int64_t)a * M + i];
        if (c0 != p0) {
#pragma unroll
            for (int c = 0; c < PW; ++c) x[c] = B[(int64_t)min(c, cn - 1) * M + i];
        }
#pragma unroll
        for (int a = 0; a < PW; ++a) v[a] = own && i > p0 + a ? v[a] : own && i == p0 + a ? 1.0 : 0.0;
        if (c0 == p0) {
#pragma unroll
            for (int c = 0; c < PW; ++c) x[c] = v[c];
        }
#pragma unroll
        for (int a = 0; a < PW; ++a)
#pragma unroll
            for (int c = 0; c < PW; ++c) acc[PW * a + c] += v[a] * x[c];
    }
    s.sums[b][wv][lane] = halve_sums<PW * PW>(acc, lane);
    __syncthreads();
    double sum = 0.0;
#pragma unroll
    for (int w = 0; w < NWR; ++w) sum += s.sums[b][w][lane];
    return sum;
}

// the panel's reflectors applied to columns c0 .. c0 + cn - 1; S, G as panel_sums
// leaves them
__device__ inline void panel_update(const TallView &T, int p0, int c0, int cn, double S, double G) {
    const int M = T.M, tid = threadIdx.x, lane = tid & 63;
    const int c = lane & 7, row = lane >> 3;
    double wl = 0.0;
#pragma unroll
    for (int l = 0; l < PW; ++l) {
        const double wf = __shfl(T.tau[p0 + l] * S, PW * l + c, 64);
        const double g = __shfl(G, PW * l + row, 64);
        if (row == l) wl = wf;
        if (row > l) S -= g * wf;
    }
    double *B = T.X + (int64_t)c0 * M;
    const double *V = T.X + (int64_t)p0 * M;
    for (int i0 = 0; i0 < M; i0 += 2 * WGR) {
        double v[2][PW], x[2][PW];
        int i[2];
        bool own[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int at = i0 + WGR * u + tid;
            i[u] = min(at, M - 1);
            own[u] = at < M && at >= p0;
#pragma unroll
            for (int a = 0; a < PW; ++a) v[u][a] = V[(int64_t)a * M + i[u]];
#pragma unroll
            for (int q = 0; q < PW; ++q) x[u][q] = B[(int64_t)min(q, cn - 1) * M + i[u]];
#pragma unroll
            for (int a = 0; a < PW; ++a)
                v[u][a] = i[u] > p0 + a ? v[u][a] : i[u] == p0 + a ? 1.0 : 0.0;
        }
#pragma unroll
        for (int q = 0; q < PW; ++q) {
#pragma unroll
            for (int a = 0; a < PW; ++a) {
                const double w = lane_value(wl, PW * a + q);
#pragma unroll
                for (int u = 0; u < 2; ++u) x[u][q] -= v[u][a] * w;
            }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if (!own[u]) continue;
#pragma unroll
            for (int q = 0; q < PW; ++q)
                if (q < cn) B[(int64_t)q * M + i[u]] = x[u][q];
        }
        if (i0 == 0 && tid >= p0 && tid < p0 + PW) {
#pragma unroll
            for (int q = 0; q < PW; ++q)
                if (q < cn) T.R[tid + LR_MAX * (c0 + q)] = x[0][q];
        }
    }
}

__device__ inline void qr_steps(const TallView &T, QrLds &s) {
    const int C = T.C;
    int b = 0;
    for (int p0 = 0; p0 < C; p0 += PW) {
        qr_panel(T, p0, min(PW, C - p0), s);
        if (p0 + PW >= C) break;
        // tau of the panel, written by the first wavefront
        __syncthreads();
        const double G = panel_sums(T, p0, p0, PW, s, b);
        b ^= 1;
        for (int c0 = p0 + PW; c0 < C; c0 += PW) {
            const int cn = min(PW, C - c0);
            const double S = panel_sums(T, p0, c0, cn, s, b);
            b ^= 1;
            panel_update(T, p0, c0, cn, S, G);
        }
    }
    for (int e = threadIdx.x; e < C * C; e += WGR) {
        const int a = e % C, c = e / C;
        if (a > c) T.R[a + LR_MAX * c] = 0.0;
    }
}

// T of Q = H_0 ... H_{C-1} = I - V T V^T (dlarft, forward, columnwise):
// T[j][j] = tau_j, T[0:j, j] = -tau_j T[0:j, 0:j] (V^T v_j)[0:j]. The Gram
// matrix V^T V is a contraction over the rows: 16 x 16 tiles on
// v_mfma_f64_16x16x4f64 (A and B operand: lane l holds V[i][l % 16] of row
// i = 4 (l / 16) + u, the same order of rows for both; D[l / 16 + 4 v][l % 16] in
// register v), sixteen rows per wavefront at a time, the wavefronts' tiles then
// added in LDS. (One pass over the rows per eight columns took 412 us, below.)
typedef double lr4_t __attribute__((ext_vector_type(4)));
struct WyLds {
    double G[LR_MAX * LD], Ts[LR_MAX * LD], part[NWR][256];
};

template <int CB>
__device__ inline void wy_steps(const TallView &T, WyLds &s) {
    constexpr int NT = CB / 16;
    const double *X = T.X;
    const int M = T.M, C = T.C;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, l16 = lane & 15, g = lane >> 4;
    lr4_t d[NT * (NT + 1) / 2];
#pragma unroll
    for (int e = 0; e < NT * (NT + 1) / 2; ++e) d[e] = lr4_t{0, 0, 0, 0};
    for (int i0 = 16 * wv; i0 < M; i0 += 16 * NWR) {
        double v[NT][4];
#pragma unroll
        for (int a = 0; a < NT; ++a) {
            const int c = 16 * a + l16;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = i0 + 4 * g + u;
                const bool below = c < C && i < M && i > c;
                const double e = X[below ? (int64_t)c * M + i : 0];
                v[a][u] = below ? e : c < C && i == c ? 1.0 : 0.0;
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            int e = 0;
#pragma unroll
            for (int b = 0; b < NT; ++b)
#pragma unroll
                for (int a = 0; a <= b; ++a, ++e)
                    d[e] = __builtin_amdgcn_mfma_f64_16x16x4f64(v[a][u], v[b][u], d[e], 0, 0, 0);
        }
    }
    {
        int e = 0;
#pragma unroll
        for (int b = 0; b < NT; ++b)
#pragma unroll
            for (int a = 0; a <= b; ++a, ++e) {
#pragma unroll
                for (int v = 0; v < 4; ++v) s.part[wv][(g + 4 * v) + 16 * l16] = d[e][v];
                __syncthreads();
                if (tid < 256) {
                    double q = 0.0;
#pragma unroll
                    for (int w = 0; w < NWR; ++w) q += s.part[w][tid];
                    s.G[16 * a + tid % 16 + LD * (16 * b + tid / 16)] = q;
                }
                __syncthreads();
            }
    }
    // the recurrence by one wavefront (C <= 64 lanes): its LDS reads and
    // writes stay in program order, so no workgroup barrier per column
    if (tid < 64) {
        for (int j = 0; j < C; ++j) {
            const double t = T.tau[j];
            if (tid < j) {
                double sacc = 0.0;
                for (int l = tid; l < j; ++l) sacc += s.Ts[tid + LD * l] * s.G[l + LD * j];
                s.Ts[tid + LD * j] = -t * sacc;
            }
            if (tid == j) s.Ts[j + LD * j] = t;
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    }
    __syncthreads();
    for (int e = tid; e < C * C; e += WGR) {
        const int a = e % C, b = e / C;
        T.T[a + LR_MAX * b] = a <= b ? s.Ts[a + LD * b] : 0.0;
    }
}

__global__ __launch_bounds__(WGR) void k_lr_qr(const LRItem *items, double *tall, double *small) {
    const LRItem it = items[blockIdx.x];
    const TallView T = tall_view(it, blockIdx.y, tall, small);
    if (T.C == 0) return;
    __shared__ union Lds {
        QrLds qr;
        WyLds wy;
        __device__ Lds() {}
    } s;
    qr_steps(T, s.qr);
    __syncthreads();
    if (T.C <= 16) wy_steps<16>(T, s.wy);
    else if (T.C <= 32) wy_steps<32>(T, s.wy);
    else wy_steps<64>(T, s.wy);
}

// entry (a, b) of the core whose SVD gives the result
__device__ inline double core_entry(int op, const LRItem &it, const double *sl, int a, int b) {
    const double *RU = sl + LR_RU, *RV = sl + LR_RV;
    switch (op) {
    case HM_LR_ADD:
    case HM_LR_SUB: {  // RU diag([S1; +-S2]) RV^T
        double g = 0.0;
        for (int t = a > b ? a : b; t < it.cu; ++t) {
            const double d = t < it.r1 ? it.S1[t]
                                       : (op == HM_LR_SUB ? -it.S2[t - it.r1] : it.S2[t - it.r1]);
            g += (RU[a + LR_MAX * t] * d) * RV[b + LR_MAX * t];
        }
        return g;
    }
    case HM_LR_MUL:
    case HM_LR_ADJMUL:  // diag(S1) M diag(S2)
        return (it.S1[a] * RU[a + LR_MAX * b]) * it.S2[b];
    case HM_LR_DMUL:  // R diag(S2)
        return RU[a + LR_MAX * b] * it.S2[b];
    case HM_LR_MULD:  // diag(S1) R^T
        return it.S1[a] * RV[b + LR_MAX * a];
    default:  // svdtrunc: R, or R^T when A^T was factored
        return it.tr ? RV[b + LR_MAX * a] : RU[a + LR_MAX * b];
    }
}

// The sum over GL lanes; every lane ends with the same bits (each addition has
// the same two operands in both partners).
template <int GL>
__device__ inline double group_sum(double v) {
    v += dpp<DPP_XOR1>(v);
    v += dpp<DPP_XOR2>(v);
    v += dpp<DPP_HALF_MIRROR>(v);
    if constexpr (GL == 16) v += dpp<DPP_MIRROR>(v);
    return v;
}

// 1/sqrt(x) and 1/x for x of the order of one: the hardware's estimate and two
// Newton steps
__device__ inline double rsqrt_unit(double x) {
    double y = __builtin_amdgcn_rsq(x);
#pragma unroll
    for (int k = 0; k < 2; ++k) y = fma(0.5 * y, fma(-x * y, y, 1.0), y);
    return y;
}
__device__ inline double rcp_unit(double x) {
    double y = __builtin_amdgcn_rcp(x);
#pragma unroll
    for (int k = 0; k < 2; ++k) y = fma(y, fma(-x, y, 1.0), y);
    return y;
}

// One-sided Jacobi (Hestenes): the columns of W (P x Q, LDS) rotated pairwise in
// round-robin order until every pair is orthogonal to 1e-15 relative; V
// accumulates the rotations. GL lanes per pair, NR rows each, held in registers
// from the dot products to the rotation. A round is one chain of dot products,
// angle, rotation, barrier; the angle is formed from the scaled pair
// (d, 2 gamma), t = 2 gamma sgn(d) / (|d| + sqrt(d^2 + 4 gamma^2)), which has one
// square root and one reciprocal in place of two divisions, a hypot and a square
// root. Cores of 10 to 32 columns: 355 -> 204 us.
template <int GL, int NR>
__device__ inline void jacobi(double *W, int LW, double *V, int LV, int P, int Q, int *flag) {
    const int tid = threadIdx.x, grp = tid / GL, l = tid % GL;
    const int Qe = Q + (Q & 1), npairs = Qe / 2;
    for (int sweep = 0; sweep < 60 && Q > 1; ++sweep) {
        if (tid == 0) *flag = 0;
        __syncthreads();
        // group 0 pairs column 0 with 1 + rd, group g > 0 the columns
        // 1 + (rd +- g) mod (Qe - 1)
        int a = grp, b = grp == 0 ? 0 : Qe - 1 - grp;
        for (int rd = 0; rd < Qe - 1; ++rd) {
            a = grp == 0 ? 0 : a == Qe - 1 ? 1 : a + 1;
            b = b == Qe - 1 ? 1 : b + 1;
            if (grp < npairs) {
                if (a < Q && b < Q) {
                    double x[NR], y[NR], vx[NR], vy[NR];
#pragma unroll
                    for (int k = 0; k < NR; ++k) {
                        const int i = l + GL * k;
                        x[k] = i < P ? W[i + LW * a] : 0.0;
                        y[k] = i < P ? W[i + LW * b] : 0.0;
                        vx[k] = i < Q ? V[i + LV * a] : 0.0;
                        vy[k] = i < Q ? V[i + LV * b] : 0.0;
                    }
                    double al = 0.0, be = 0.0, ga = 0.0;
#pragma unroll
                    for (int k = 0; k < NR; ++k) {
                        al += x[k] * x[k];
                        be += y[k] * y[k];
                        ga += x[k] * y[k];
                    }
                    al = group_sum<GL>(al);
                    be = group_sum<GL>(be);
                    ga = group_sum<GL>(ga);
                    // |ga| > 1e-15 sqrt(al be), squared where that neither
                    // over- nor underflows
                    const double ab = al * be;
                    const bool rot = ga != 0.0 && (ab > 1e-250 ? ga * ga > 1e-30 * ab
                                                              : fabs(ga) > 1e-15 * sqrt(ab));
                    if (rot) {
                        if (l == 0) *flag = 1;
                        double d = be - al, g2 = 2.0 * ga;
                        const int e = -__builtin_amdgcn_frexp_exp(fmax(fabs(d), fabs(g2)));
                        d = ldexp(d, e);
                        g2 = ldexp(g2, e);
                        const double ss = d * d + g2 * g2, h = ss * rsqrt_unit(ss);
                        const double t = copysign(1.0, d) * g2 * rcp_unit(fabs(d) + h);
                        const double c = rsqrt_unit(1.0 + t * t), s = c * t;
#pragma unroll
                        for (int k = 0; k < NR; ++k) {
                            const int i = l + GL * k;
                            if (i < P) {
                                W[i + LW * a] = c * x[k] - s * y[k];
                                W[i + LW * b] = s * x[k] + c * y[k];
                            }
                            if (i < Q) {
                                V[i + LV * a] = c * vx[k] - s * vy[k];
                                V[i + LV * b] = s * vx[k] + c * vy[k];
                            }
                        }
                    }
                }
            }
            __syncthreads();
        }
        const int f = *flag;
        __syncthreads();
        if (!f) break;
    }
}

// SVD of the core by one-sided Jacobi: W (P x Q, Q <= P) = G, or G^T when G has
// more columns than rows. Then S = column norms sorted descending,
// U = W V-columns / S, getrank. Writes S, SU (p x min), SV (q x min), the
// rank, and the result's S.
__global__ __launch_bounds__(WG) void k_lr_svd(int op, const LRItem *items, double *small) {
    const LRItem it = items[blockIdx.x];
    double *sl = small + it.small;
    const int p = it.p, q = it.q, tid = threadIdx.x;
    const bool trn = q > p;
    const int P = trn ? q : p, Q = trn ? p : q;
    // W: P x Q (ld P + 1), V: Q x Q (ld Q + 1), nrm: Q
    extern __shared__ double dyn[];
    const int LW = P + 1, LV = Q + 1;
    double *W = dyn, *V = dyn + LW * Q, *nrm = V + LV * Q;
    __shared__ int flag;
    for (int e = tid; e < p * q; e += WG) {
        const int a = e % p, b = e / p;
        const double g = core_entry(op, it, sl, a, b);
        if (trn) W[b + LW * a] = g;
        else W[a + LW * b] = g;
    }
    for (int e = tid; e < Q * Q; e += WG) {
        const int a = e % Q, b = e / Q;
        V[a + LV * b] = a == b ? 1.0 : 0.0;
    }
    __syncthreads();
    if (P <= 32) jacobi<16, 2>(W, LW, V, LV, P, Q, &flag);
    else if (Q <= 32) jacobi<16, 4>(W, LW, V, LV, P, Q, &flag);
    else jacobi<8, 8>(W, LW, V, LV, P, Q, &flag);
    for (int j = tid; j < Q; j += WG) {
        double s = 0.0;
        for (int i = 0; i < P; ++i) s += W[i + LW * j] * W[i + LW * j];
        nrm[j] = sqrt(s);
    }
    __syncthreads();
    double *Uo = sl + (trn ? LR_SV : LR_SU);  // P x Q
    double *Vo = sl + (trn ? LR_SU : LR_SV);  // Q x Q
    double *S = sl + LR_S;
    for (int j = tid; j < Q; j += WG) {
        const double sj = nrm[j];
        int pos = 0;
        for (int k = 0; k < Q; ++k) pos += (nrm[k] > sj) || (nrm[k] == sj && k < j);
        S[pos] = sj;
        for (int i = 0; i < P; ++i) Uo[i + LR_MAX * pos] = sj > 0.0 ? W[i + LW * j] / sj : 0.0;
        for (int i = 0; i < Q; ++i) Vo[i + LR_MAX * pos] = V[i + LV * j];
    }
    __syncthreads();
    if (tid == 0) {
        // getrank, src/LowRankMatrix.jl:70-80: tol = length(S) * eps(S[1])
        const double tol = (double)Q * (nextafter(S[0], INFINITY) - S[0]);
        int r = Q;
        while (r >= 1 && !(S[r - 1] > tol)) --r;
        sl[LR_RANK] = (double)r;
    }
    __syncthreads();
    const int r = (int)sl[LR_RANK];
    for (int c = tid; c < r; c += WG) it.So[c] = S[c];
}

// W = T (V^T [B; 0]) (C x r) for out = Q [B; 0] = [B; 0] - V W, with B the
// first r columns of SU or SV (C x r) and V unit lower triangular in its top
// C rows. W goes to the RU / RV place of the small slot (the SVD has used
// R by now), where k_lr_applyq reads it with wave-uniform addresses.
__global__ __launch_bounds__(WG) void k_lr_wz(const LRItem *items, double *tall, double *small,
                                              int ldw) {
    const LRItem it = items[blockIdx.x];
    const int side = blockIdx.y;
    const TallView T = tall_view(it, side, tall, small);
    if (T.C == 0) return;
    double *sl = small + it.small;
    const double *B = sl + (side ? LR_SV : LR_SU);
    double *Wg = sl + (side ? LR_RV : LR_RU);
    const int M = T.M, C = T.C, tid = threadIdx.x;
    const int R = (int)sl[LR_RANK];
    const double *X = T.X;
    // the top C rows of V, B's first r columns and T staged in LDS (one
    // batch of loads each) before the products; ldw = the call's largest C
    // plus one (dynamic LDS, 4 * C * ldw doubles)
    extern __shared__ double wzs[];
    const int LW = ldw, CW = ldw - 1;
    double *Z = wzs, *Vt = Z + CW * LW, *Bs = Vt + CW * LW, *Ts = Bs + CW * LW;
    for (int e = tid; e < C * C; e += WG) {
        const int i = e % C, a = e / C;
        Vt[i + LW * a] = X[(int64_t)a * M + i];
        Ts[i + LW * a] = T.T[i + LR_MAX * a];
    }
    for (int e = tid; e < C * R; e += WG) {
        const int i = e % C, k = e / C;
        Bs[i + LW * k] = B[i + LR_MAX * k];
    }
    __syncthreads();
    for (int e = tid; e < C * R; e += WG) {
        const int a = e % C, k = e / C;
        double z = Bs[a + LW * k];  // V[a][a] = 1, V[i][a] stored below
        for (int i = a + 1; i < C; ++i) z += Vt[i + LW * a] * Bs[i + LW * k];
        Z[a + LW * k] = z;
    }
    __syncthreads();
    for (int e = tid; e < C * R; e += WG) {
        const int a = e % C, k = e / C;
        double wv = 0.0;
        for (int l = a; l < C; ++l) wv += Ts[a + LW * l] * Z[l + LW * k];
        Wg[k + LR_MAX * a] = wv;  // row a contiguous: W[a][0..r)
    }
}

// out[i, :] = [B; 0][i, :] - V[i, :] W, one thread per row i, with RB
// accumulators (RB >= rank R); W (C x r) is read at wave-uniform addresses,
// and the reflector entries of four columns are loaded before their products
template <int RB>
__device__ inline void applyq_row(const double *X, int M, int C, int R, int i, const double *Wg,
                                  const double *B, double *out) {
    double acc[RB];
#pragma unroll
    for (int k = 0; k < RB; ++k) acc[k] = 0.0;
    for (int t0 = 0; t0 < C; t0 += 4) {
        double v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            // V[i][t]: 0 above the diagonal, 1 on it, stored below
            const int t = t0 + u;
            const bool below = t < C && i > t && i < M;
            const double x = X[below ? (int64_t)t * M + i : 0];
            v[u] = below ? x : (t < C && i == t ? 1.0 : 0.0);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (t0 + u < C) {
                const double *wr = Wg + LR_MAX * (t0 + u);
#pragma unroll
                for (int k = 0; k < RB; ++k) acc[k] += v[u] * wr[k];
            }
        }
    }
    if (i < M) {
#pragma unroll
        for (int k = 0; k < RB; ++k)
            if (k < R) out[i + (int64_t)M * k] = (i < C ? B[i + LR_MAX * k] : 0.0) - acc[k];
    }
}

__global__ __launch_bounds__(WG) void k_lr_applyq(const LRItem *items, double *tall,
                                                  double *small) {
    const LRItem it = items[blockIdx.x];
    const int side = blockIdx.y;
    const TallView T = tall_view(it, side, tall, small);
    if (T.C == 0) return;
    const double *sl = small + it.small;
    const double *B = sl + (side ? LR_SV : LR_SU);
    const double *Wg = sl + (side ? LR_RV : LR_RU);
    double *out = side ? it.Vo : it.Uo;
    const int M = T.M, C = T.C;
    const int R = (int)sl[LR_RANK];
    const int i = blockIdx.z * WG + threadIdx.x;
    if (blockIdx.z * WG >= M) return;
    // W's columns past R hold finite values (or zeros) and are not stored
    if (R <= 16) applyq_row<16>(T.X, M, C, R, i, Wg, B, out);
    else if (R <= 32) applyq_row<32>(T.X, M, C, R, i, Wg, B, out);
    else applyq_row<LR_MAX>(T.X, M, C, R, i, Wg, B, out);
}

__global__ void k_lr_ranks(const LRItem *items, int64_t count, const double *small,
                           int64_t *rank) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < count) rank[t] = (int64_t)small[items[t].small + LR_RANK];
}

}  // namespace

hipError_t hmx_lowrank_run(int op, const LRItem *items, int64_t count, double *tall,
                           double *small, int64_t *rank, int64_t max_rows, int64_t lds_svd,
                           int64_t max_c, hipStream_t s) {
    if (count <= 0) return hipSuccess;
    const unsigned n = (unsigned)count;
    const unsigned rowblk = (unsigned)((max_rows + WG - 1) / WG);
    if (op == HM_LR_ADD || op == HM_LR_SUB || op == HM_LR_SVDTRUNC)
        k_lr_pack<<<dim3(n, 2, rowblk < 64 ? rowblk : 64), WG, 0, s>>>(op, items, tall);
    if (op == HM_LR_DMUL || op == HM_LR_MULD)
        k_lr_gemm<LR_MAX><<<dim3(n, 2, rowblk), WG, 0, s>>>(op, 0, items, tall, small);
    if (op == HM_LR_MUL || op == HM_LR_ADJMUL) {
        k_lr_gram<<<n, WG, 0, s>>>(op, items, small);
    } else {
        k_lr_qr<<<dim3(n, 2), WGR, 0, s>>>(items, tall, small);
    }
    k_lr_svd<<<n, WG, sizeof(double) * (size_t)lds_svd, s>>>(op, items, small);
    if (op != HM_LR_MUL && op != HM_LR_ADJMUL) {
        const int ldw = (int)max_c + 1;
        const size_t wz_bytes = sizeof(double) * 4 * (size_t)max_c * ldw;
        if (wz_bytes > 65536)
            (void)hipFuncSetAttribute((const void *)k_lr_wz,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)wz_bytes);
        k_lr_wz<<<dim3(n, 2), WG, wz_bytes, s>>>(items, tall, small, ldw);
        k_lr_applyq<<<dim3(n, 2, rowblk), WG, 0, s>>>(items, tall, small);
    }
    k_lr_gemm<LR_MAX><<<dim3(n, 2, rowblk), WG, 0, s>>>(op, 1, items, tall, small);
    k_lr_ranks<<<(n + 255) / 256, 256, 0, s>>>(items, count, small, rank);
    return hipGetLastError();
}
