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

// One point of a set (a's at A, b's at B, three doubles each) added to the
// sums of the centroids.
__device__ static inline void add_centroid(const double *A, const double *B, double ca[3], double cb[3])
{
#pragma unroll
    for (int d = 0; d < 3; d++) {
        ca[d] += A[d];
        cb[d] += B[d];
    }
}

// ... to the correlation X.
__device__ static inline void add_correlation(const double *A, const double *B, const double ca[3],
                                              const double cb[3], double X[3][3])
{
    double u[3], v[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        u[d] = A[d] - ca[d];
        v[d] = B[d] - cb[d];
    }
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
        for (int k = 0; k < 3; k++) X[j][k] += v[j] * u[k];
}

// ... to the squared residuals of rotation R.
__device__ static inline void add_residual(const double *A, const double *B, const double ca[3], const double cb[3],
                                           const double R[3][3], double &e)
{
    double u[3], v[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        u[d] = A[d] - ca[d];
        v[d] = B[d] - cb[d];
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double ra = R[d][0] * u[0] + R[d][1] * u[1] + R[d][2] * u[2];
        const double r = v[d] - ra;
        e += r * r;
    }
}

// The point's gradients, in place of the point (scale: the RMSD's gradient over
// n * rmsd).
__device__ static inline void to_gradient(double *A, double *B, const double ca[3], const double cb[3],
                                          const double R[3][3], double scale)
{
    double u[3], v[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        u[d] = A[d] - ca[d];
        v[d] = B[d] - cb[d];
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
        // (R^T B_i)_d and (R A_i)_d
        const double rtb = R[0][d] * v[0] + R[1][d] * v[1] + R[2][d] * v[2];
        const double ra = R[d][0] * u[0] + R[d][1] * u[1] + R[d][2] * u[2];
        A[d] = scale * (u[d] - rtb);
        B[d] = scale * (v[d] - ra);
    }
}

// The sums above over a set of n points, which `each` hands to its argument in
// order.
template <class E>
__device__ static inline void centroids(int n, E each, double ca[3], double cb[3])
{
#pragma unroll
    for (int d = 0; d < 3; d++) {
        ca[d] = 0.0;
        cb[d] = 0.0;
    }
    each([&](double *A, double *B) { add_centroid(A, B, ca, cb); });
#pragma unroll
    for (int d = 0; d < 3; d++) {
        ca[d] /= (double)n;
        cb[d] /= (double)n;
    }
}

template <class E>
__device__ static inline void correlate(E each, const double ca[3], const double cb[3], double X[3][3])
{
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
        for (int k = 0; k < 3; k++) X[j][k] = 0.0;
    each([&](double *A, double *B) { add_correlation(A, B, ca, cb, X); });
}

template <class E>
__device__ static inline double residual(int n, E each, const double ca[3], const double cb[3], const double R[3][3])
{
    double e = 0.0;
    each([&](double *A, double *B) { add_residual(A, B, ca, cb, R, e); });
    return sqrt(e / (double)n);
}

// One wave per tile of RG_SETS consecutive sets (one set per lane), a lane
// summing its set point by point: the same operations in the same order
// whichever way the points reach it.
//
// k_rmsd_*<false>, up to RG_FEW_TILES tiles: one wave for each of the 1,024
// SIMDs, which do not compete for the caches. Both arrays of the tile in LDS (37
// KB) where its points fit, else every lane reads its set from global memory,
// RG_FAR points in flight. 64 sets of 8 points, forward and backward: 14 + 11 us;
// of 200: 77 + 128 us (in chunks 374 + 351).
//
// k_rmsd_*<true>, more tiles: bound by the waves per SIMD (the rotation is a chain of some hundreds
// of dependent FP64 operations) and by memory, so one array in LDS (18 KB) and
// two waves per SIMD, whose lanes reading 64 sets at once would thrash the L1 (1.25 M
// sets of 16 points: 1.05 + 2.0 ms):
//   sets of at most RG_REG points, together at most RG_CAP: a through LDS into
//     registers, then b, which stays there; the gradients leave the same way. In
//     the forward pass larger sets may be among them, whose lanes read the
//     array that is not in LDS from global memory. 1 M sets of 3 to 12 points, forward
//     and backward: 0.31 ms, against 0.49 with both arrays in LDS (0.25 at the
//     rate of a copy);
//   else up to RG_ROUNDS rounds of as many sets as LDS holds of both arrays (a
//     set too large for that alone, from global memory): 416,666 sets of 24 points
//     (four rounds) 0.31 + 0.29 ms, in chunks 0.39 + 0.40;
//   else RG_CHUNK points of every set at a time, once for each of the sums
//     (centroids, correlation, residuals or gradients), the next chunk's loads
//     in flight: all lanes work, and the rotation is done once. 312,500 sets of 32
//     points 0.39 + 0.45 ms, in six rounds 0.46 + 0.45; 50,000 of 200 points
//     and up in rounds of one to three lanes: 7 ms and more.
#define RG_SETS 64
#define RG_REG 12    // points of a set held in registers
#define RG_CAP (RG_SETS * RG_REG)   // points of one array held in LDS
#define RG_LOADS (3 * RG_CAP / RG_SETS)
#define RG_NEAR 2    // points in flight from LDS
#define RG_FAR 4     // ... from global memory
#define RG_FEW_TILES 1024
#define RG_ROUNDS 4
#define RG_CHUNK 5   // 15 doubles a set: an odd stride, so that the lanes' reads spread over the banks
#define RG_TEAM 16   // lanes that load a set's chunk
#define RG_ROWS (RG_SETS * RG_TEAM / JAM_WAVE)

struct RmsdChunks {
    double a[RG_SETS * 3 * RG_CHUNK], b[RG_SETS * 3 * RG_CHUNK];
    long long at[RG_SETS], len[RG_SETS];   // each set's first double and number of doubles
};

template <bool MANY>
union RmsdLds {
    double l[3 * RG_CAP * (MANY ? 1 : 2)];
    RmsdChunks c;
};

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

// m doubles of a and of b into LDS, the loads of N * RG_SETS of each in flight
template <int N>
__device__ static inline void stage_both(const double *a, const double *b, int m, int lane, double *la, double *lb)
{
    for (int q = 0; q < m; q += N * RG_SETS) {
        double ra[N], rb[N];
        tile_load(a + q, m - q, lane, ra);
        tile_load(b + q, m - q, lane, rb);
        tile_store(ra, m - q, lane, la + q);
        tile_store(rb, m - q, lane, lb + q);
    }
    wave_sync();
}

// Both arrays of the tile: a's points of this lane's set (n of them from p)
// into A where they are at most RG_REG, b's into LDS; `between` runs while a's
// are there.
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
        for (int d = 0; d < 3; d++) A[3 * i + d] = i < n && n <= RG_REG ? l[3 * (p + i) + d] : 0.0;
    between();
    wave_sync();
    tile_store(rb, m, lane, l);
    wave_sync();
}

// The points of a set in registers (A) and LDS (B), n <= RG_REG.
template <class F>
__device__ static inline void each_staged(int n, double (&A)[3 * RG_REG], double *B, F point)
{
#pragma unroll
    for (int i = 0; i < RG_REG; i++)
        if (i < n) point(A + 3 * i, B + 3 * i);
}

// The points of a set at A and B, the loads of U points in flight.
template <int U, class F>
__device__ static inline void each_at(int n, const double *A, const double *B, F point)
{
#pragma unroll U
    for (int i = 0; i < n; i++) {
        double x[3], y[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            x[d] = A[3 * i + d];
            y[d] = B[3 * i + d];
        }
        point(x, y);
    }
}

// The same, what point() makes of them going to GA and GB (each may be null;
// they may be A and B).
template <int U, class F>
__device__ static inline void each_into(int n, const double *A, const double *B, double *GA, double *GB, F point)
{
    int i = 0;
    each_at<U>(n, A, B, [&](double *x, double *y) {
        point(x, y);
#pragma unroll
        for (int d = 0; d < 3; d++) {
            if (GA) GA[3 * i + d] = x[d];
            if (GB) GB[3 * i + d] = y[d];
        }
        i++;
    });
}

// Doubles [3c, 3c + 15) of every set of the tile, RG_TEAM lanes a set.
__device__ static inline void chunk_load(const RmsdChunks &S, const double *src, long long c, int lane,
                                         double (&r)[RG_ROWS])
{
    const int i = lane % RG_TEAM;
#pragma unroll
    for (int u = 0; u < RG_ROWS; u++) {
        const int j = u * (JAM_WAVE / RG_TEAM) + lane / RG_TEAM;
        const bool in = i < 3 * RG_CHUNK && 3 * c + i < S.len[j];
        r[u] = in ? src[S.at[j] + 3 * c + i] : 0.0;
    }
}

__device__ static inline void chunk_put(double *l, int lane, const double (&r)[RG_ROWS])
{
    const int i = lane % RG_TEAM;
#pragma unroll
    for (int u = 0; u < RG_ROWS; u++)
        if (i < 3 * RG_CHUNK) l[(u * (JAM_WAVE / RG_TEAM) + lane / RG_TEAM) * 3 * RG_CHUNK + i] = r[u];
}

__device__ static inline void chunk_store(const RmsdChunks &S, const double *l, long long c, int lane, double *dst)
{
    const int i = lane % RG_TEAM;
#pragma unroll
    for (int u = 0; u < RG_ROWS; u++) {
        const int j = u * (JAM_WAVE / RG_TEAM) + lane / RG_TEAM;
        if (i < 3 * RG_CHUNK && 3 * c + i < S.len[j]) dst[S.at[j] + 3 * c + i] = l[j * 3 * RG_CHUNK + i];
    }
}

// point() for every point of the lanes' sets (n of the lane's, `most` of the
// largest), a chunk at a time; after(c) when all lanes are done with chunk c.
// The whole wave calls it.
template <class F, class G>
__device__ static inline void each_chunked(const double *a, const double *b, RmsdChunks &S, int n, int most, int lane,
                                           F point, G after)
{
    double ra[RG_ROWS], rb[RG_ROWS];
    chunk_load(S, a, 0, lane, ra);
    chunk_load(S, b, 0, lane, rb);
    for (long long c = 0; c < most; c += RG_CHUNK) {
        wave_sync();
        chunk_put(S.a, lane, ra);
        chunk_put(S.b, lane, rb);
        wave_sync();
        if (c + RG_CHUNK < most) {
            chunk_load(S, a, c + RG_CHUNK, lane, ra);
            chunk_load(S, b, c + RG_CHUNK, lane, rb);
        }
#pragma unroll
        for (int i = 0; i < RG_CHUNK; i++)
            if (c + i < n) point(S.a + 3 * (RG_CHUNK * lane + i), S.b + 3 * (RG_CHUNK * lane + i));
        after(c);
    }
    wave_sync();
}

// The table of the lanes' sets ([p0, p0 + n) of each), and the largest n.
__device__ static inline int chunk_table(RmsdChunks &S, int64_t p0, int n, int lane)
{
    S.at[lane] = 3 * (long long)p0;
    S.len[lane] = 3 * (long long)max(n, 0);
    wave_sync();
    int most = n;
#pragma unroll
    for (int sh = JAM_WAVE / 2; sh >= 1; sh >>= 1) most = max(most, __shfl_xor(most, sh, JAM_WAVE));
    return most;
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

// The sets [g0, g1) of the tile that one round takes, and their points [q0, q1):
// those that fit half the buffer, or one set alone, where that is larger. The
// lanes' ranges never descend, so that those that fit are the first ones.
__device__ static inline bool tile_round(int64_t p0, int64_t p1, int g0, int lane, int &g1, int64_t &q0, int64_t &q1)
{
    q0 = __shfl(p0, g0, JAM_WAVE);
    const int fit = __popcll(ballot(lane >= g0 && p1 - q0 <= RG_CAP / 2));
    g1 = g0 + max(fit, 1);
    q1 = __shfl(p1, g1 - 1, JAM_WAVE);
    // within the buffer whatever the offsets
    if (fit) q1 = q1 < q0 ? q0 : (q1 > q0 + RG_CAP / 2 ? q0 + RG_CAP / 2 : q1);
    return fit > 0;
}

// Whether the tile takes at most `most` rounds.
__device__ static inline bool few_rounds(int64_t p0, int64_t p1, int lane, int most)
{
    int g1 = 0;
    int64_t q0, q1;
    for (int k = 0; k < most && g1 < RG_SETS; k++) (void)tile_round(p0, p1, g1, lane, g1, q0, q1);
    return g1 >= RG_SETS;
}

// RMSD and rotation of a set of n points.
template <class E>
__device__ static inline double rmsd_of(int n, E each, double R[3][3])
{
    double ca[3], cb[3], X[3][3];
    centroids(n, each, ca, cb);
    correlate(each, ca, cb, X);
    optimal_rotation(X, R);
    return residual(n, each, ca, cb, R);
}

// Set s owns points [off[s], off[s+1]) of a and b, 3 doubles per point.
template <bool MANY>
__global__ void __launch_bounds__(RG_SETS, MANY ? 2 : 1) k_rmsd_fwd(const double *a, const double *b,
                                                                   const int64_t *off, long long n_sets,
                                                                   long long n_points, double *rmsd, double *rot)
{
    __shared__ RmsdLds<MANY> S;
    const int lane = threadIdx.x;
    const long long s = (long long)blockIdx.x * RG_SETS + lane;
    int64_t P0, P1, p0, p1;
    tile_ranges(off, n_sets, n_points, s, P0, P1, p0, p1);
    const int n = (int)(p1 - p0);
    const bool fits = P1 - P0 <= RG_CAP;
    const int at = 3 * (int)(p0 - P0), m = (int)(3 * (P1 - P0));   // where it fits
    double r = 0.0, R[3][3];
    if (!MANY) {
        if (fits) {
            const double *A = S.l + at, *B = A + 3 * RG_CAP;
            stage_both<12>(a + 3 * P0, b + 3 * P0, m, lane, S.l, S.l + 3 * RG_CAP);
            if (n > 0) r = rmsd_of(n, [&](auto point) { each_at<RG_NEAR>(n, A, B, point); }, R);
        } else if (n > 0) {
            r = rmsd_of(n, [&](auto point) { each_at<RG_FAR>(n, a + 3 * p0, b + 3 * p0, point); }, R);
        }
    } else if (fits) {
        double A[3 * RG_REG], ca[3], cb[3], X[3][3];
        const bool large = n > RG_REG;
        stage_tile(a + 3 * P0, b + 3 * P0, m, lane, at / 3, n, S.l, A, [&] {
            if (!large) return;
            auto each = [&](auto point) { each_at<RG_FAR>(n, S.l + at, b + 3 * p0, point); };
            centroids(n, each, ca, cb);
            correlate(each, ca, cb, X);
        });
        auto each = [&](auto point) { each_staged(n, A, S.l + at, point); };
        if (!large) {
            centroids(n, each, ca, cb);
            correlate(each, ca, cb, X);
        }
        if (n > 0) {
            optimal_rotation(X, R);
            r = large ? residual(n, [&](auto point) { each_at<RG_FAR>(n, a + 3 * p0, S.l + at, point); }, ca, cb, R)
                      : residual(n, each, ca, cb, R);
        }
    } else if (few_rounds(p0, p1, lane, RG_ROUNDS)) {
        for (int g0 = 0, g1; g0 < RG_SETS; g0 = g1) {
            int64_t q0, q1;
            const double *A = a + 3 * p0, *B = b + 3 * p0;
            const bool staged = tile_round(p0, p1, g0, lane, g1, q0, q1);
            bool now = lane >= g0 && lane < g1 && n > 0;
            if (staged) {
                stage_both<RG_LOADS / 2>(a + 3 * q0, b + 3 * q0, (int)(3 * (q1 - q0)), lane, S.l,
                                         S.l + 3 * RG_CAP / 2);
                now = now && p0 >= q0 && p1 <= q1;
                A = S.l + 3 * (int)(p0 - q0);
                B = A + 3 * RG_CAP / 2;
            }
            if (now) r = rmsd_of(n, [&](auto point) { each_at<RG_FAR>(n, A, B, point); }, R);
            wave_sync();
        }
    } else {
        const int most = chunk_table(S.c, p0, n, lane);
        r = rmsd_of(n, [&](auto point) { each_chunked(a, b, S.c, n, most, lane, point, [](long long) {}); }, R);
        if (n <= 0) r = 0.0;
    }
    if (s >= n_sets) return;
    rmsd[s] = r;
    double *rt = rot ? rot + 9 * s : nullptr;
    if (rt)
#pragma unroll
        for (int q = 0; q < 9; q++) rt[q] = n > 0 ? R[q / 3][q % 3] : (q % 4 == 0) ? 1.0 : 0.0;
}

template <bool MANY>
__global__ void __launch_bounds__(RG_SETS, MANY ? 2 : 1) k_rmsd_bwd(const double *a, const double *b,
                                                                   const int64_t *off, long long n_sets,
                                                                   long long n_points, const double *rmsd,
                                                                   const double *rot, const double *grad_rmsd,
                                                                   double *grad_a, double *grad_b)
{
    __shared__ RmsdLds<MANY> S;
    const int lane = threadIdx.x;
    const long long s = (long long)blockIdx.x * RG_SETS + lane;
    int64_t P0, P1, p0, p1;
    tile_ranges(off, n_sets, n_points, s, P0, P1, p0, p1);
    const int n = (int)(p1 - p0);   // 0 past the last set
    const bool fits = P1 - P0 <= RG_CAP;
    const int at = 3 * (int)(p0 - P0), m = (int)(3 * (P1 - P0));   // where it fits
    const double r = n > 0 ? rmsd[s] : 0.0, g = n > 0 ? grad_rmsd[s] : 0.0;
    bool zero = true;
    double ca[3], cb[3], R[3][3], scale = 0.0;
    // what gradient() needs; rot: the optimal rotations of the forward pass, or
    // null to compute them again
    auto prepare = [&](auto each) {
        zero = !(r > 0.0) || g == 0.0;
        scale = g / ((double)n * r);
        centroids(n, each, ca, cb);
        if (rot) {
            if (n > 0)
#pragma unroll
                for (int q = 0; q < 9; q++) R[q / 3][q % 3] = rot[9 * s + q];
        } else {
            double X[3][3];
            correlate(each, ca, cb, X);
            optimal_rotation(X, R);
        }
    };
    auto gradient = [&](double *A, double *B) {
        if (zero) {
#pragma unroll
            for (int d = 0; d < 3; d++) A[d] = B[d] = 0.0;
        } else {
            to_gradient(A, B, ca, cb, R, scale);
        }
    };
    const double *Ag = a + 3 * p0, *Bg = b + 3 * p0;
    if (MANY && fits && ballot(n > RG_REG) == 0ull) {
        double A[3 * RG_REG], *B = S.l + at;
        stage_tile(a + 3 * P0, b + 3 * P0, m, lane, at / 3, n, S.l, A, [] {});
        if (n > 0) {
            prepare([&](auto point) { each_staged(n, A, B, point); });
            each_staged(n, A, B, gradient);
        }
        // b's gradients from LDS, then a's through it
        wave_sync();
        if (grad_b)
            for (int q = lane; q < m; q += RG_SETS) grad_b[3 * P0 + q] = S.l[q];
        wave_sync();
        if (!grad_a) return;
        each_staged(n, A, B, [](double *x, double *l) {
#pragma unroll
            for (int d = 0; d < 3; d++) l[d] = x[d];
        });
        wave_sync();
        for (int q = lane; q < m; q += RG_SETS) grad_a[3 * P0 + q] = S.l[q];
    } else if (!MANY && !fits) {
        if (n > 0) {
            prepare([&](auto point) { each_at<RG_FAR>(n, Ag, Bg, point); });
            each_into<RG_FAR>(n, Ag, Bg, grad_a ? grad_a + 3 * p0 : nullptr, grad_b ? grad_b + 3 * p0 : nullptr,
                              gradient);
        }
    } else if (!MANY || few_rounds(p0, p1, lane, RG_ROUNDS)) {
        // rounds; without MANY one, of the whole tile
        constexpr int HALF = 3 * RG_CAP / (MANY ? 2 : 1), NEAR = MANY ? RG_FAR : RG_NEAR;
        for (int g0 = 0, g1 = RG_SETS; g0 < RG_SETS; g0 = g1) {
            int64_t q0 = P0, q1 = P1;
            if (MANY && !tile_round(p0, p1, g0, lane, g1, q0, q1)) {
                if (lane == g0) {   // larger than the buffer
                    prepare([&](auto point) { each_at<RG_FAR>(n, Ag, Bg, point); });
                    each_into<RG_FAR>(n, Ag, Bg, grad_a ? grad_a + 3 * p0 : nullptr,
                                      grad_b ? grad_b + 3 * p0 : nullptr, gradient);
                }
                continue;
            }
            const int k = (int)(3 * (q1 - q0));
            stage_both<MANY ? RG_LOADS / 2 : 12>(a + 3 * q0, b + 3 * q0, k, lane, S.l, S.l + HALF);
            if (lane >= g0 && lane < g1 && n > 0 && p0 >= q0 && p1 <= q1) {
                // gradients replace the points in LDS
                double *A = S.l + 3 * (int)(p0 - q0), *B = A + HALF;
                prepare([&](auto point) { each_at<NEAR>(n, A, B, point); });
                each_into<NEAR>(n, A, B, A, B, gradient);
            }
            wave_sync();
            for (int q = lane; q < k; q += RG_SETS) {
                if (grad_a) grad_a[3 * q0 + q] = S.l[q];
                if (grad_b) grad_b[3 * q0 + q] = S.l[HALF + q];
            }
            wave_sync();
        }
    } else {
        const int most = chunk_table(S.c, p0, n, lane);
        prepare([&](auto point) { each_chunked(a, b, S.c, n, most, lane, point, [](long long) {}); });
        each_chunked(a, b, S.c, n, most, lane, gradient, [&](long long c) {
            wave_sync();
            if (grad_a) chunk_store(S.c, S.c.a, c, lane, grad_a);
            if (grad_b) chunk_store(S.c, S.c.b, c, lane, grad_b);
        });
    }
}

}  // namespace jam
