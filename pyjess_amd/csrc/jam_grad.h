// jam_grad.h -- differentiable superposition RMSD of many point-set pairs.
//
// rmsd = sqrt(E / n), E = sum_i |B_i - R A_i|^2, A and B the centred points
// and R the proper rotation that minimises E (the least-squares
// superposition of a onto b: the quantity of Superposition_rmsd,
// include/jess/super.pxd:1-14). With X = sum_i B_i A_i^T = U S V^T,
// R = U diag(1, 1, det(U) det(V)) V^T.
//
// R is computed from a one-sided Jacobi SVD of X (Hestenes: plane rotations
// of the columns until they are orthogonal; Demmel & Veselic, "Jacobi's
// method is more accurate than QR", 1992), which keeps the small singular
// values -- nearly planar or nearly collinear sets -- to high relative
// accuracy, with u3 = u1 x u2 so that the frame is proper even when
// sigma3 = 0. E is then summed from the residuals directly: no cancellation,
// and only second order in the error of R because R minimises E. (The
// search's hit decisions use the reference's eigenvalue formula instead,
// jam_super.h; the two agree to rounding on well-conditioned sets.)
//
// Gradient: dE/dR vanishes at the optimum (envelope theorem) and centring
// drops out of the chain rule because centred points sum to zero, so
//     d rmsd / d a_i = (A_i - R^T B_i) / (n rmsd),
//     d rmsd / d b_i = (B_i - R A_i) / (n rmsd);
// taken as zero where rmsd = 0.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>

#include "jam_wave.h"

namespace jam {

// Optimal proper rotation R (row-major 3x3) for the correlation X.
__device__ static inline void optimal_rotation(const double X[3][3], double R[3][3])
{
    double W[3][3], V[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            W[i][j] = X[i][j];
            V[i][j] = (i == j) ? 1.0 : 0.0;
        }
    for (int sweep = 0; sweep < 16; sweep++) {
        bool rotated = false;
#pragma unroll
        for (int r = 0; r < 3; r++) {
            const int p = (r == 2) ? 1 : 0;
            const int q = (r == 0) ? 1 : 2;
            double al = 0.0, be = 0.0, ga = 0.0;
#pragma unroll
            for (int j = 0; j < 3; j++) {
                al += W[j][p] * W[j][p];
                be += W[j][q] * W[j][q];
                ga += W[j][p] * W[j][q];
            }
            if (ga == 0.0 || fabs(ga) <= 1e-15 * sqrt(al * be)) continue;
            const double ze = (be - al) / (2.0 * ga);
            double t = 1.0 / (fabs(ze) + sqrt(1.0 + ze * ze));
            if (ze < 0.0) t = -t;
            const double c = 1.0 / sqrt(1.0 + t * t);
            const double s = c * t;
#pragma unroll
            for (int j = 0; j < 3; j++) {
                const double wp = W[j][p], wq = W[j][q];
                W[j][p] = c * wp - s * wq;
                W[j][q] = s * wp + c * wq;
                const double vp = V[j][p], vq = V[j][q];
                V[j][p] = c * vp - s * vq;
                V[j][q] = s * vp + c * vq;
            }
            rotated = true;
        }
        if (!rotated) break;
    }
    // columns of W are U S: order by singular value
    double sg[3];
#pragma unroll
    for (int i = 0; i < 3; i++) sg[i] = sqrt(W[0][i] * W[0][i] + W[1][i] * W[1][i] + W[2][i] * W[2][i]);
    // (by exchanging columns: an index into the registers would be memory)
    auto order = [&](int i, int j) {
        if (!(sg[j] > sg[i])) return;
        const double x = sg[i];
        sg[i] = sg[j];
        sg[j] = x;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const double w = W[k][i], v = V[k][i];
            W[k][i] = W[k][j];
            W[k][j] = w;
            V[k][i] = V[k][j];
            V[k][j] = v;
        }
    };
    order(0, 1);
    order(1, 2);
    order(0, 1);
    double u1[3], u2[3], u3[3], v1[3], v2[3], v3[3];
#pragma unroll
    for (int j = 0; j < 3; j++) {
        u1[j] = sg[0] > 0.0 ? W[j][0] / sg[0] : (j == 0 ? 1.0 : 0.0);
        u2[j] = W[j][1];
        v1[j] = V[j][0];
        v2[j] = V[j][1];
        v3[j] = V[j][2];
    }
    if (sg[1] > 0.0) {
#pragma unroll
        for (int j = 0; j < 3; j++) u2[j] /= sg[1];
    } else {
        // rank <= 1: any unit vector orthogonal to u1 (the axis of u1's
        // smallest component, made orthogonal)
        const bool y = fabs(u1[1]) < fabs(u1[0]);
        const bool z = fabs(u1[2]) < (y ? fabs(u1[1]) : fabs(u1[0]));
        const double e[3] = {!y && !z ? 1.0 : 0.0, y && !z ? 1.0 : 0.0, z ? 1.0 : 0.0};
        const double dp = u1[0] * e[0] + u1[1] * e[1] + u1[2] * e[2];
        double w[3] = {e[0] - dp * u1[0], e[1] - dp * u1[1], e[2] - dp * u1[2]};
        const double nw = sqrt(w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
#pragma unroll
        for (int j = 0; j < 3; j++) u2[j] = w[j] / nw;
    }
    u3[0] = u1[1] * u2[2] - u1[2] * u2[1];
    u3[1] = u1[2] * u2[0] - u1[0] * u2[2];
    u3[2] = u1[0] * u2[1] - u1[1] * u2[0];
    const double detv = v1[0] * (v2[1] * v3[2] - v2[2] * v3[1]) - v1[1] * (v2[0] * v3[2] - v2[2] * v3[0]) +
                        v1[2] * (v2[0] * v3[1] - v2[1] * v3[0]);
    const double sgn = detv < 0.0 ? -1.0 : 1.0;
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
        for (int k = 0; k < 3; k++) R[j][k] = u1[j] * v1[k] + u2[j] * v2[k] + sgn * u3[j] * v3[k];
}

// Centroids and the correlation X of points [0, n) of A and B.
__device__ static inline void centre_and_correlate(int n, const double *A, const double *B, double ca[3],
                                                   double cb[3], double X[3][3])
{
#pragma unroll
    for (int d = 0; d < 3; d++) {
        ca[d] = 0.0;
        cb[d] = 0.0;
    }
    for (int i = 0; i < n; i++)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            ca[d] += A[3 * i + d];
            cb[d] += B[3 * i + d];
        }
#pragma unroll
    for (int d = 0; d < 3; d++) {
        ca[d] /= (double)n;
        cb[d] /= (double)n;
    }
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
        for (int k = 0; k < 3; k++) X[j][k] = 0.0;
    for (int i = 0; i < n; i++) {
        double u[3], v[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            u[d] = A[3 * i + d] - ca[d];
            v[d] = B[3 * i + d] - cb[d];
        }
#pragma unroll
        for (int j = 0; j < 3; j++)
#pragma unroll
            for (int k = 0; k < 3; k++) X[j][k] += v[j] * u[k];
    }
}

// One set: RMSD from the residuals of rotation R.
__device__ static inline double residual_rmsd(int n, const double *A, const double *B, const double ca[3],
                                              const double cb[3], const double R[3][3])
{
    double e = 0.0;
    for (int i = 0; i < n; i++) {
        double u[3], v[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            u[d] = A[3 * i + d] - ca[d];
            v[d] = B[3 * i + d] - cb[d];
        }
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const double ra = R[d][0] * u[0] + R[d][1] * u[1] + R[d][2] * u[2];
            const double r = v[d] - ra;
            e += r * r;
        }
    }
    return sqrt(e / (double)n);
}

// One set: the gradient of g * rmsd, written to GA / GB (which may alias A /
// B: every point is read before its gradient is written). rot: the set's
// optimal rotation from the forward pass, or null to compute it again.
__device__ __attribute__((always_inline)) static inline void rmsd_grad_one(int n, const double *A, const double *B,
                                                                           double r, double g, const double *rot,
                                                                           double *GA, double *GB)
{
    if (!(r > 0.0) || g == 0.0) {
        for (int q = 0; q < 3 * n; q++) {
            if (GA) GA[q] = 0.0;
            if (GB) GB[q] = 0.0;
        }
        return;
    }
    double ca[3], cb[3], R[3][3];
    if (rot) {
        // centroids only: the rotation is the forward pass's
#pragma unroll
        for (int d = 0; d < 3; d++) {
            ca[d] = 0.0;
            cb[d] = 0.0;
        }
        for (int i = 0; i < n; i++)
#pragma unroll
            for (int d = 0; d < 3; d++) {
                ca[d] += A[3 * i + d];
                cb[d] += B[3 * i + d];
            }
#pragma unroll
        for (int d = 0; d < 3; d++) {
            ca[d] /= (double)n;
            cb[d] /= (double)n;
        }
#pragma unroll
        for (int j = 0; j < 3; j++)
#pragma unroll
            for (int k = 0; k < 3; k++) R[j][k] = rot[3 * j + k];
    } else {
        double X[3][3];
        centre_and_correlate(n, A, B, ca, cb, X);
        optimal_rotation(X, R);
    }
    const double scale = g / ((double)n * r);
    for (int i = 0; i < n; i++) {
        double u[3], v[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            u[d] = A[3 * i + d] - ca[d];
            v[d] = B[3 * i + d] - cb[d];
        }
        double ga[3], gb[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            // (R^T B_i)_d and (R A_i)_d
            const double rtb = R[0][d] * v[0] + R[1][d] * v[1] + R[2][d] * v[2];
            const double ra = R[d][0] * u[0] + R[d][1] * u[1] + R[d][2] * u[2];
            ga[d] = scale * (u[d] - rtb);
            gb[d] = scale * (v[d] - ra);
        }
#pragma unroll
        for (int d = 0; d < 3; d++) {
            if (GA) GA[3 * i + d] = ga[d];
            if (GB) GB[3 * i + d] = gb[d];
        }
    }
}

// One wave per tile of RG_SETS consecutive sets (one set per lane), its points
// moved by coalesced loads and stores through one LDS buffer. A tile of sets of
// up to RG_REG points that fits the buffer (RG_CAP points of one array) goes
// through it an array at a time: a, which every lane takes into registers, then
// b, which stays in LDS; the gradients leave the same way (in the forward pass
// larger sets may be among them). Any other tile goes in rounds of as many sets as the buffer holds of both arrays (RG_CAP / 2
// points); a set too large for that is read from global memory by its lane.
//
// Bound by latency: the rotation is a chain of some hundreds of dependent FP64
// operations per lane, so what counts is the waves per SIMD: one array in LDS
// (18 KB) instead of two (37 KB) makes them two instead of one, and the loads
// of both arrays are all in flight before the first LDS store. 1 M sets of 3 to
// 12 points, forward and backward: 0.49 -> 0.31 ms (0.25 ms at the rate of a
// copy); 400,000 sets of 24 points: 1.27 -> 0.67 ms.
#define RG_SETS 64
#define RG_CAP 768   // points per tile held in LDS (12 per set on average)
#define RG_REG 12    // points of a set held in registers
#define RG_LOADS (3 * RG_CAP / RG_SETS)

// m doubles of src (m <= N * RG_SETS), one in RG_SETS to each lane
template <int N>
__device__ static inline void tile_load(const double *src, int m, int lane, double (&r)[N])
{
#pragma unroll
    for (int u = 0; u < N; u++) {
        const int q = lane + RG_SETS * u;
        r[u] = q < m ? src[q] : 0.0;
    }
}

template <int N>
__device__ static inline void tile_store(const double (&r)[N], int m, int lane, double *l)
{
#pragma unroll
    for (int u = 0; u < N; u++) {
        const int q = lane + RG_SETS * u;
        if (q < m) l[q] = r[u];
    }
}

// m doubles of a and of b (m <= 3 * RG_CAP / 2) into LDS
__device__ static inline void stage_pair(const double *a, const double *b, int m, int lane, double *la, double *lb)
{
    double ra[RG_LOADS / 2], rb[RG_LOADS / 2];
    tile_load(a, m, lane, ra);
    tile_load(b, m, lane, rb);
    tile_store(ra, m, lane, la);
    tile_store(rb, m, lane, lb);
}

// Both arrays of the tile: a's points of this lane's set (n of them from p)
// into A, b's into LDS; `between` runs while a's are there.
template <class F>
__device__ static inline void stage_tile(const double *a, const double *b, int m, int lane, int p, int n, double *l,
                                         double (&A)[3 * RG_REG], F between)
{
    double ra[RG_LOADS], rb[RG_LOADS];
    tile_load(a, m, lane, ra);
    tile_load(b, m, lane, rb);
    tile_store(ra, m, lane, l);
    wave_sync();
#pragma unroll
    for (int i = 0; i < RG_REG; i++)
#pragma unroll
        for (int d = 0; d < 3; d++) A[3 * i + d] = (i < n && n <= RG_REG) ? l[3 * (p + i) + d] : 0.0;
    between();
    wave_sync();
    tile_store(rb, m, lane, l);
    wave_sync();
}

// The functions above (whose operations and order these keep) for A in
// registers, n <= RG_REG.
__device__ static inline void centroids_reg(int n, const double (&A)[3 * RG_REG], const double *B, double ca[3],
                                            double cb[3])
{
#pragma unroll
    for (int d = 0; d < 3; d++) {
        ca[d] = 0.0;
        cb[d] = 0.0;
    }
#pragma unroll
    for (int i = 0; i < RG_REG; i++) {
        if (i < n) {
#pragma unroll
            for (int d = 0; d < 3; d++) {
                ca[d] += A[3 * i + d];
                cb[d] += B[3 * i + d];
            }
        }
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
        ca[d] /= (double)n;
        cb[d] /= (double)n;
    }
}

__device__ static inline void correlate_reg(int n, const double (&A)[3 * RG_REG], const double *B, const double ca[3],
                                            const double cb[3], double X[3][3])
{
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
        for (int k = 0; k < 3; k++) X[j][k] = 0.0;
#pragma unroll
    for (int i = 0; i < RG_REG; i++) {
        if (i < n) {
            double u[3], v[3];
#pragma unroll
            for (int d = 0; d < 3; d++) {
                u[d] = A[3 * i + d] - ca[d];
                v[d] = B[3 * i + d] - cb[d];
            }
#pragma unroll
            for (int j = 0; j < 3; j++)
#pragma unroll
                for (int k = 0; k < 3; k++) X[j][k] += v[j] * u[k];
        }
    }
}

__device__ static inline double residual_reg(int n, const double (&A)[3 * RG_REG], const double *B, const double ca[3],
                                             const double cb[3], const double R[3][3])
{
    double e = 0.0;
#pragma unroll
    for (int i = 0; i < RG_REG; i++) {
        if (i < n) {
            double u[3], v[3];
#pragma unroll
            for (int d = 0; d < 3; d++) {
                u[d] = A[3 * i + d] - ca[d];
                v[d] = B[3 * i + d] - cb[d];
            }
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const double ra = R[d][0] * u[0] + R[d][1] * u[1] + R[d][2] * u[2];
                const double r = v[d] - ra;
                e += r * r;
            }
        }
    }
    return sqrt(e / (double)n);
}

// gradients replace A and B
__device__ static inline void rmsd_grad_reg(int n, double (&A)[3 * RG_REG], double *B, double r, double g,
                                            const double *rot)
{
    if (!(r > 0.0) || g == 0.0) {
#pragma unroll
        for (int q = 0; q < 3 * RG_REG; q++) A[q] = 0.0;
        for (int q = 0; q < 3 * n; q++) B[q] = 0.0;
        return;
    }
    double ca[3], cb[3], R[3][3];
    centroids_reg(n, A, B, ca, cb);
    if (rot) {
#pragma unroll
        for (int j = 0; j < 3; j++)
#pragma unroll
            for (int k = 0; k < 3; k++) R[j][k] = rot[3 * j + k];
    } else {
        double X[3][3];
        correlate_reg(n, A, B, ca, cb, X);
        optimal_rotation(X, R);
    }
    const double scale = g / ((double)n * r);
#pragma unroll
    for (int i = 0; i < RG_REG; i++) {
        if (i < n) {
            double u[3], v[3];
#pragma unroll
            for (int d = 0; d < 3; d++) {
                u[d] = A[3 * i + d] - ca[d];
                v[d] = B[3 * i + d] - cb[d];
            }
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const double rtb = R[0][d] * v[0] + R[1][d] * v[1] + R[2][d] * v[2];
                const double ra = R[d][0] * u[0] + R[d][1] * u[1] + R[d][2] * u[2];
                A[3 * i + d] = scale * (u[d] - rtb);
                B[3 * i + d] = scale * (v[d] - ra);
            }
        }
    }
}

// Range of set s, clamped into [lo, hi]: with valid offsets (off[0] = 0,
// never decreasing, off[n_sets] = n_points) this is [off[s], off[s+1]);
// malformed offsets give meaningless values, never an access outside a and b.
__device__ static inline void set_range(const int64_t *off, long long s, int64_t lo, int64_t hi, int64_t &p0,
                                        int64_t &p1)
{
    int64_t x = off[s], y = off[s + 1];
    x = x < lo ? lo : (x > hi ? hi : x);
    y = y < x ? x : (y > hi ? hi : y);
    p0 = x;
    p1 = y;
}

// The tile's points [P0, P1) and the lane's set's [p0, p1) (empty for a lane
// past the last set).
__device__ static inline void tile_ranges(const int64_t *off, long long n_sets, long long n_points, long long s,
                                          int64_t &P0, int64_t &P1, int64_t &p0, int64_t &p1)
{
    const long long s0 = (long long)blockIdx.x * RG_SETS;
    const long long s1 = s0 + RG_SETS < n_sets ? s0 + RG_SETS : n_sets;
    int64_t q0, q1;
    set_range(off, s0, 0, n_points, P0, q0);
    set_range(off, s1 - 1, P0, n_points, q1, P1);
    p0 = p1 = P1;
    if (s < s1) set_range(off, s, P0, P1, p0, p1);
}

// The sets [g0, g1) of the tile that one round takes: its first point, and g1
// (g0 where the first set alone is too large). The lanes' ranges never
// descend, so that those that fit are the first ones.
__device__ static inline int64_t tile_round(int64_t p0, int64_t p1, int g0, int lane, int &g1)
{
    const int64_t q0 = __shfl(p0, g0, JAM_WAVE);
    g1 = g0 + __popcll(ballot(lane >= g0 && p1 - q0 <= RG_CAP / 2));
    return q0;
}

// The round's end: the last point of its last set, within the buffer whatever
// the offsets.
__device__ static inline int64_t round_end(int64_t p1, int64_t q0, int g1)
{
    const int64_t q1 = __shfl(p1, g1 - 1, JAM_WAVE);
    return q1 < q0 ? q0 : (q1 > q0 + RG_CAP / 2 ? q0 + RG_CAP / 2 : q1);
}

// Set s owns points [off[s], off[s+1]) of a and b, 3 doubles per point.
__global__ void __launch_bounds__(RG_SETS, 2) k_rmsd_fwd(const double *a, const double *b, const int64_t *off,
                                                         long long n_sets, long long n_points, double *rmsd,
                                                         double *rot)
{
    __shared__ double l[3 * RG_CAP];
    const int lane = threadIdx.x;
    const long long s = (long long)blockIdx.x * RG_SETS + lane;
    int64_t P0, P1, p0, p1;
    tile_ranges(off, n_sets, n_points, s, P0, P1, p0, p1);
    const int n = (int)(p1 - p0);
    double r = 0.0;
    double *rt = rot ? rot + 9 * s : nullptr;
    double ca[3], cb[3], X[3][3], R[3][3];
    if (P1 - P0 <= RG_CAP) {
        // larger sets than the registers hold read the array that is not in
        // LDS from global memory, where the tile's loads have just been
        const int at = (int)(p0 - P0);
        const bool small = n <= RG_REG;
        double A[3 * RG_REG];
        stage_tile(a + 3 * P0, b + 3 * P0, (int)(3 * (P1 - P0)), lane, at, n, l, A, [&] {
            if (!small) centre_and_correlate(n, l + 3 * at, b + 3 * p0, ca, cb, X);
        });
        if (small) {
            centroids_reg(n, A, l + 3 * at, ca, cb);
            correlate_reg(n, A, l + 3 * at, ca, cb, X);
        }
        if (n > 0) {
            optimal_rotation(X, R);
            r = small ? residual_reg(n, A, l + 3 * at, ca, cb, R)
                      : residual_rmsd(n, a + 3 * p0, l + 3 * at, ca, cb, R);
        }
    } else {
        for (int g0 = 0, g1; g0 < RG_SETS; g0 = g1) {
            const int64_t q0 = tile_round(p0, p1, g0, lane, g1);
            const double *A = a + 3 * p0, *B = b + 3 * p0;
            bool now = lane == g0 && n > 0;
            if (g1 > g0) {
                const int64_t q1 = round_end(p1, q0, g1);
                stage_pair(a + 3 * q0, b + 3 * q0, (int)(3 * (q1 - q0)), lane, l, l + 3 * RG_CAP / 2);
                wave_sync();
                now = lane >= g0 && lane < g1 && n > 0 && p0 >= q0 && p1 <= q1;
                A = l + 3 * (int)(p0 - q0);
                B = A + 3 * RG_CAP / 2;
            } else {
                g1++;   // larger than the buffer
            }
            if (now) {
                centre_and_correlate(n, A, B, ca, cb, X);
                optimal_rotation(X, R);
                r = residual_rmsd(n, A, B, ca, cb, R);
            }
            wave_sync();
        }
    }
    if (s >= n_sets) return;
    rmsd[s] = r;
    if (rt)
#pragma unroll
        for (int q = 0; q < 9; q++) rt[q] = n > 0 ? R[q / 3][q % 3] : (q % 4 == 0) ? 1.0 : 0.0;
}

__global__ void __launch_bounds__(RG_SETS, 2) k_rmsd_bwd(const double *a, const double *b, const int64_t *off,
                                                         long long n_sets, long long n_points, const double *rmsd,
                                                         const double *rot, const double *grad_rmsd, double *grad_a,
                                                         double *grad_b)
{
    __shared__ double l[3 * RG_CAP];
    const int lane = threadIdx.x;
    const long long s = (long long)blockIdx.x * RG_SETS + lane;
    int64_t P0, P1, p0, p1;
    tile_ranges(off, n_sets, n_points, s, P0, P1, p0, p1);
    const int n = (int)(p1 - p0);
    const bool mine = n > 0;   // never past the last set
    const double *rt = rot ? rot + 9 * s : nullptr;
    if (P1 - P0 <= RG_CAP && ballot(n > RG_REG) == 0ull) {
        const int at = (int)(p0 - P0), m = (int)(3 * (P1 - P0));
        double A[3 * RG_REG];
        stage_tile(a + 3 * P0, b + 3 * P0, m, lane, at, n, l, A, [] {});
        if (mine) rmsd_grad_reg(n, A, l + 3 * at, rmsd[s], grad_rmsd[s], rt);
        // b's gradients from LDS, then a's through it
        wave_sync();
        if (grad_b)
            for (int q = lane; q < m; q += RG_SETS) grad_b[3 * P0 + q] = l[q];
        wave_sync();
        if (!grad_a) return;
        if (mine)
#pragma unroll
            for (int i = 0; i < RG_REG; i++)
#pragma unroll
                for (int d = 0; d < 3; d++)
                    if (i < n) l[3 * (at + i) + d] = A[3 * i + d];
        wave_sync();
        for (int q = lane; q < m; q += RG_SETS) grad_a[3 * P0 + q] = l[q];
        return;
    }
    for (int g0 = 0, g1; g0 < RG_SETS; g0 = g1) {
        const int64_t q0 = tile_round(p0, p1, g0, lane, g1);
        if (g1 == g0) {
            // larger than the buffer
            if (lane == g0)
                rmsd_grad_one(n, a + 3 * p0, b + 3 * p0, rmsd[s], grad_rmsd[s], rt,
                              grad_a ? grad_a + 3 * p0 : nullptr, grad_b ? grad_b + 3 * p0 : nullptr);
            g1++;
            continue;
        }
        const int64_t q1 = round_end(p1, q0, g1);
        const int m = (int)(3 * (q1 - q0));
        double *la = l, *lb = l + 3 * RG_CAP / 2;
        stage_pair(a + 3 * q0, b + 3 * q0, m, lane, la, lb);
        wave_sync();
        if (lane >= g0 && lane < g1 && mine && p0 >= q0 && p1 <= q1) {
            // gradients replace the points in LDS
            const int at = 3 * (int)(p0 - q0);
            rmsd_grad_one(n, la + at, lb + at, rmsd[s], grad_rmsd[s], rt, la + at, lb + at);
        }
        wave_sync();
        for (int q = lane; q < m; q += RG_SETS) {
            if (grad_a) grad_a[3 * q0 + q] = la[q];
            if (grad_b) grad_b[3 * q0 + q] = lb[q];
        }
        wave_sync();
    }
}

}  // namespace jam
