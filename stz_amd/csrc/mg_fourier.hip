// mg_fourier.hip -- direct solve of the projection's top-level operator.
//
// qs_multi's operator (qs_multi.hh:30-50, qs_multi.cc:31-54) does not depend
// on x, which is periodic, and away from the two wall rows not on y either.
// A discrete Fourier transform along x therefore leaves, for each mode
// k = 0..M/2, a block tridiagonal Toeplitz system over the N = n - 1 interior
// rows whose 2x2 blocks are real once the transverse velocity is written
// v = i v':
//     Cd w_{j-1} + B w_j + Cu w_{j+1} = f_j,   w = (u, v'),  Cd = Cu^T.
// With D the limit of the elimination D -> B - Cd D^{-1} Cu the system factors
// as T = L U + E1 P E1^T, L and U bidiagonal with constant blocks and
// P = B - D acting on the first row only, so one solve is a forward and a
// backward recurrence with constant coefficients F = -Cd D^{-1} and
// E = -D^{-1} Cu = F^T, and the first row's rank-two term:
//     g_j = f_j + F g_{j-1},  y_j = D^{-1} g_j + E y_{j+1}   (y = M^{-1} f)
//     w_1 = (I + G P)^{-1} y_1,  w = M^{-1}(f - E1 P w_1),   G = (M^{-1})_11.
// Constant coefficients make both recurrences scans: each lane of a mode's
// workgroup runs P rows, and the carries combine through F^P, F^2P, F^4P, ...
// Per mode the host forms D, F, the powers and P (I + G P)^{-1} in extended
// precision (the limit by cyclic reduction, which converges quadratically;
// mode 0 in closed form: D = -Cu, F = I).  In FP64 the result is at the
// rounding floor: the residual is 1e-16 of the source on every size from 8^2
// to 1024^2, so one application replaces all V-cycles of a solve.
//
// Three launches:
//   forward   R rows per workgroup: u + i v of a row as one complex signal
//             (in a step the source is formed here), an in-LDS Stockham
//             transform, the two real signals' modes separated on the way out
//   modes     one workgroup per mode, the column in LDS
//   inverse   R rows per workgroup, back to (u, v)
// Each is bound by its memory passes and, in front of them, by one chain of
// loads, barriers and stores: at 1024^2 19.4 (64 bytes a node, source
// included), 13.3 and 10.7 us (32 bytes a node each; the copy rate gives 13,
// 6.6 and 6.6), where the V-cycles of a step took 250 to 1200; at 2048^2 79, 38
// and 38 us (53, 26 and 26).
// The spectrum is kept mode-major, S[k][j] of 32 bytes (u, v' complex), a
// column padded to four rows, so the mode launch reads and writes whole
// columns and a row workgroup touches R * 32 contiguous bytes per mode.
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>
#include <vector>

#include "batch.h"
#include "device.h"
#include "mg.h"
#include "mg_node.h"

namespace stz {

// ---------------------------------------------------------------------------
// the row transform
// ---------------------------------------------------------------------------
// rows per workgroup R with 128 threads each: four where that leaves a
// workgroup per CU (their 128-byte pieces of the spectrum are whole cache
// lines), else two.  A row's result does not depend on R.
constexpr int kRowThreads = 128;

struct alignas(16) cplx { double x, y; };

__device__ __forceinline__ static cplx operator+(const cplx &a, const cplx &b) { return {a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ static cplx operator-(const cplx &a, const cplx &b) { return {a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ static cplx cmul(const cplx &a, const cplx &b) {
    return {fmav(a.x, b.x, -(a.y * b.y)), fmav(a.x, b.y, a.y * b.x)};
}
__device__ __forceinline__ static cplx mul_mi(const cplx &a) { return {a.y, -a.x}; }  // -i a

// LDS position of element i: one 16-byte slot in nine is skipped, so that
// the transform's strided writes (strides 4, 8) spread over the banks
__host__ __device__ constexpr int fpad(int i) { return i + (i >> 3); }

// forward DFTs of R values in place (e^{-2 pi i / R})
template <int R> __device__ __forceinline__ static void dft(cplx (&x)[R]);
template <> __device__ __forceinline__ void dft<2>(cplx (&x)[2]) {
    const cplx a = x[0], b = x[1];
    x[0] = a + b;
    x[1] = a - b;
}
template <> __device__ __forceinline__ void dft<3>(cplx (&x)[3]) {
    const double s = 0.86602540378443864676;  // sqrt(3)/2
    const cplx t = x[1] + x[2], d = x[1] - x[2], a = x[0];
    const cplx c = {fmav(-0.5, t.x, a.x), fmav(-0.5, t.y, a.y)};
    x[0] = a + t;
    x[1] = {fmav(s, d.y, c.x), fmav(-s, d.x, c.y)};
    x[2] = {fmav(-s, d.y, c.x), fmav(s, d.x, c.y)};
}
template <> __device__ __forceinline__ void dft<4>(cplx (&x)[4]) {
    const cplx a = x[0] + x[2], b = x[0] - x[2], c = x[1] + x[3], d = mul_mi(x[1] - x[3]);
    x[0] = a + c;
    x[1] = b + d;
    x[2] = a - c;
    x[3] = b - d;
}
template <> __device__ __forceinline__ void dft<5>(cplx (&x)[5]) {
    const double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;  // cos 2 pi/5, 4 pi/5
    const double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;   // sin
    const cplx a = x[0], p = x[1] + x[4], q = x[2] + x[3], m = x[1] - x[4], n = x[2] - x[3];
    const cplx u = {fmav(c2, q.x, fmav(c1, p.x, a.x)), fmav(c2, q.y, fmav(c1, p.y, a.y))};
    const cplx v = {fmav(c1, q.x, fmav(c2, p.x, a.x)), fmav(c1, q.y, fmav(c2, p.y, a.y))};
    const cplx f = {fmav(s1, m.x, s2 * n.x), fmav(s1, m.y, s2 * n.y)};
    const cplx g = {fmav(s2, m.x, -(s1 * n.x)), fmav(s2, m.y, -(s1 * n.y))};
    x[0] = a + p + q;
    x[1] = {u.x + f.y, u.y - f.x};
    x[4] = {u.x - f.y, u.y + f.x};
    x[2] = {v.x + g.y, v.y - g.x};
    x[3] = {v.x - g.y, v.y + g.x};
}
template <> __device__ __forceinline__ void dft<8>(cplx (&x)[8]) {
    const double h = 0.70710678118654752440;
    cplx e[4] = {x[0], x[2], x[4], x[6]}, o[4] = {x[1], x[3], x[5], x[7]};
    dft<4>(e);
    dft<4>(o);
    const cplx o1 = {h * (o[1].x + o[1].y), h * (o[1].y - o[1].x)};
    const cplx o2 = mul_mi(o[2]);
    const cplx o3 = {h * (o[3].y - o[3].x), -h * (o[3].x + o[3].y)};
    x[0] = e[0] + o[0];
    x[4] = e[0] - o[0];
    x[1] = e[1] + o1;
    x[5] = e[1] - o1;
    x[2] = e[2] + o2;
    x[6] = e[2] - o2;
    x[3] = e[3] + o3;
    x[7] = e[3] - o3;
}

// Twiddles of a stage after radices of product L: entry (q - 1) L + k of the
// stage's part of the table, which starts at L - 1 (the parts of the stages
// before it), so a wave's loads of one q are consecutive.
template <int RX, int L, int Q> struct Twiddles { cplx w[Q][RX > 1 ? RX - 1 : 1]; };

// radix of the stage after a product of L, for the lengths known at compile
// time: 8 while that leaves a multiple of 4, then 4 and at most one 2
__host__ __device__ constexpr int fixed_radix(int left) {
    return left % 8 == 0 && left != 16 ? 8 : (left % 4 == 0 ? 4 : (left > 1 ? 2 : 1));
}

template <int M, int R, int RX, int L>
__device__ __forceinline__ static auto load_twiddles(const cplx *__restrict__ tw) {
    constexpr int NT = kRowThreads * R, NBF = R * (M / RX), Q = (NBF + NT - 1) / NT;
    Twiddles<RX, L, Q> t;
    if constexpr (RX > 1) {
#pragma unroll
        for (int b = 0; b < Q; b++) {
            const int k = ((threadIdx.x + NT * b) % (M / RX)) % L;
#pragma unroll
            for (int q = 1; q < RX; q++) t.w[b][q - 1] = tw[L - 1 + (q - 1) * L + k];
        }
    }
    return t;
}

// One Stockham stage for R rows of M values in `buf`, in place, and those
// after it.  Every butterfly of a thread is in registers between the two
// barriers, which is why M is a compile-time constant here; the next stage's
// twiddles are loaded before them.
template <int M, int R, int RX, int L, int Q>
__device__ __forceinline__ static void stages_fixed(cplx *buf, const cplx *__restrict__ tw,
                                                    const Twiddles<RX, L, Q> &w) {
    constexpr int NT = kRowThreads * R, NBF = R * (M / RX);
    cplx x[Q][RX];
#pragma unroll
    for (int b = 0; b < Q; b++) {
        const int t = threadIdx.x + NT * b;
        if (NBF % NT == 0 || t < NBF) {
            const int row = t / (M / RX), idx = t % (M / RX);
#pragma unroll
            for (int q = 0; q < RX; q++) x[b][q] = buf[row * fpad(M) + fpad(idx + q * (M / RX))];
            if (L > 1)
#pragma unroll
                for (int q = 1; q < RX; q++) x[b][q] = cmul(x[b][q], w.w[b][q - 1]);
            dft<RX>(x[b]);
        }
    }
    constexpr int LN = L * RX, RN = fixed_radix(M / LN);
    const auto next = load_twiddles<M, R, RN, LN>(tw);
    __syncthreads();
#pragma unroll
    for (int b = 0; b < Q; b++) {
        const int t = threadIdx.x + NT * b;
        if (NBF % NT == 0 || t < NBF) {
            const int row = t / (M / RX), idx = t % (M / RX);
            const int o = (idx / L) * (L * RX) + idx % L;
#pragma unroll
            for (int q = 0; q < RX; q++) buf[row * fpad(M) + fpad(o + q * L)] = x[b][q];
        }
    }
    __syncthreads();
    if constexpr (RN > 1) stages_fixed<M, R>(buf, tw, next);
}

// t / d for 0 <= t < 2^16 with inv = 1.0f / d: (t + 1/2) / d is at least
// 1 / (2 d) from a whole number, more than the product's rounding
__device__ __forceinline__ static int small_div(int t, float inv) { return (int)(((float)t + 0.5f) * inv); }

// any length: one stage from `in` to `out`, radix RX
template <int RX, int R>
__device__ __forceinline__ static void stage_any(const cplx *in, cplx *out, const cplx *__restrict__ tw, int M, int L) {
    constexpr int NT = kRowThreads * R;
    const int P = fpad(M), nb = M / RX;
    const float inb = 1.0f / nb, il = 1.0f / L;
    for (int t = threadIdx.x; t < R * nb; t += NT) {
        const int row = small_div(t, inb), idx = t - row * nb, k = idx - L * small_div(idx, il);
        cplx x[RX];
#pragma unroll
        for (int q = 0; q < RX; q++) x[q] = in[row * P + fpad(idx + q * nb)];
        if (L > 1)
#pragma unroll
            for (int q = 1; q < RX; q++) x[q] = cmul(x[q], tw[L - 1 + (q - 1) * L + k]);
        dft<RX>(x);
        const int o = (idx - k) * RX + k;
#pragma unroll
        for (int q = 0; q < RX; q++) out[row * P + fpad(o + q * L)] = x[q];
    }
}

// the same for a prime r without a butterfly above.  In place in `in`, the
// twiddles, and of each pair of inputs p, r - p the sum and the difference;
// then a thread per pair of outputs q, r - q, which share
//     x_0 + sum_p (x_p + x_{r-p}) cos(2 pi p q / r)  and
//     sum_p (x_p - x_{r-p}) sin(2 pi p q / r),
// a quarter of the multiplications of a sum per output.  rt: the r roots of
// unity e^{-2 pi i m / r}, in LDS.  608 columns (19 x 32), a source
// launch of 317 rows: 22.5 us as a plain sum per output with its roots from
// memory, 14.2 this way.
template <int R>
__device__ __forceinline__ static void stage_prime(cplx *in, cplx *out, const cplx *__restrict__ tw, const cplx *rt,
                                                   int M, int L, int r) {
    constexpr int NT = kRowThreads * R;
    const int P = fpad(M), nb = M / r, h = r / 2;
    const float inb = 1.0f / nb, il = 1.0f / L, ih = 1.0f / h, ih1 = 1.0f / (h + 1);
    for (int t = threadIdx.x; t < R * nb * h; t += NT) {
        const int u = small_div(t, inb), idx = t - u * nb, row = small_div(u, ih), p = 1 + u - row * h;
        const int k = idx - L * small_div(idx, il);
        cplx *lo = in + row * P + fpad(idx + p * nb), *hi = in + row * P + fpad(idx + (r - p) * nb);
        cplx x = *lo, y = *hi;
        if (L > 1) {
            x = cmul(x, tw[L - 1 + (p - 1) * L + k]);
            y = cmul(y, tw[L - 1 + (r - p - 1) * L + k]);
        }
        *lo = x + y;
        *hi = x - y;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < R * nb * (h + 1); t += NT) {
        const int u = small_div(t, inb), idx = t - u * nb, row = small_div(u, ih1), q = u - row * (h + 1);
        const int k = idx - L * small_div(idx, il);
        const cplx *x = in + row * P;
        cplx c = x[fpad(idx)], f = {0, 0};
        int m = 0;
#pragma unroll 3
        for (int p = 1; p <= h; p++) {
            m += q;
            if (m >= r) m -= r;
            const cplx w = rt[m], a = x[fpad(idx + p * nb)], b = x[fpad(idx + (r - p) * nb)];
            c = {fmav(w.x, a.x, c.x), fmav(w.x, a.y, c.y)};
            f = {fmav(w.y, b.x, f.x), fmav(w.y, b.y, f.y)};  // minus the sine sum
        }
        cplx *o = out + row * P;
        const int e = (idx - k) * r + k;
        o[fpad(e + q * L)] = {c.x - f.y, c.y + f.x};
        if (q > 0) o[fpad(e + (r - q) * L)] = {c.x + f.y, c.y - f.x};
    }
}

// transform the R rows in LDS; returns where the result is
template <int MT, int R>
__device__ __forceinline__ static cplx *transform_rows(const FourierArgs &a, cplx *buf) {
    const cplx *tw = reinterpret_cast<const cplx *>(a.tw);
    if constexpr (MT > 0) {
        stages_fixed<MT, R>(buf, tw, load_twiddles<MT, R, fixed_radix(MT), 1>(tw));
        return buf;
    } else {
        const cplx *root = tw + a.M;
        cplx *in = buf, *out = buf + R * fpad(a.M);
        int L = 1;
        for (int s = 0; s < a.nst; s++) {
            const int r = a.radix[s];
            if (r == 8) stage_any<8, R>(in, out, tw, a.M, L);
            else if (r == 4) stage_any<4, R>(in, out, tw, a.M, L);
            else if (r == 2) stage_any<2, R>(in, out, tw, a.M, L);
            else if (r == 3) stage_any<3, R>(in, out, tw, a.M, L);
            else if (r == 5) stage_any<5, R>(in, out, tw, a.M, L);
            else {
                cplx *rt = buf + 2 * R * fpad(a.M);
                for (int m = threadIdx.x; m < r; m += kRowThreads * R) rt[m] = root[m * (a.M / r)];
                // stage_prime's own barrier lies between these stores and their use
                stage_prime<R>(in, out, tw, rt, a.M, L, r);
            }
            __syncthreads();
            cplx *t = in;
            in = out;
            out = t;
            L *= r;
        }
        return in;
    }
}

// the solved value of wall node (i, row 0 or n): its row holds the diagonal only
__device__ __forceinline__ static cplx wall_node(const FourierArgs &a, const cplx *src, int i, int j) {
    const cplx s = src[(size_t)i + (size_t)a.M * j];
    return {a.wix * s.x, a.wiy * s.y};
}

// the wall velocity's part of the row next to it, moved to the right-hand
// side: c, l, r the wall node below (above) and its neighbours, sg 1 (-1)
__device__ __forceinline__ static cplx less_wall(const FourierArgs &a, const cplx &v, const cplx &c, const cplx &l,
                                                 const cplx &r, double sg) {
    return {v.x - fmav(a.cxx, c.x, sg * (a.cxy * (l.y - r.y))), v.y - fmav(a.cyy, c.y, sg * (a.cxy * (l.x - r.x)))};
}

// transform the R rows in `buf` (interior rows j0 ..) and store their modes:
// twice those of u and of v' = -i v, from those of u + i v
template <int MT, int R>
__device__ __forceinline__ static void store_modes(const FourierArgs &a, cplx *buf, int j0) {
    constexpr int NT = kRowThreads * R;
    const int M = MT > 0 ? MT : a.M, N = a.N, K = M / 2 + 1;
    const cplx *c = transform_rows<MT, R>(a, buf);
    double2 *S = reinterpret_cast<double2 *>(a.S);
    for (int t = threadIdx.x; t < R * K; t += NT) {
        const int row = t % R, k = t / R, j = j0 - 1 + row;
        if (j >= N) continue;
        const cplx p = c[row * fpad(M) + fpad(k)], q = c[row * fpad(M) + fpad(k == 0 ? 0 : M - k)];
        double2 *o = S + 2 * ((size_t)k * a.NP + j);
        o[0] = make_double2(p.x + q.x, p.y - q.y);
        o[1] = make_double2(q.x - p.x, -p.y - q.y);
    }
}

// forward launch body: interior rows 1 + R * blk .. of the source
template <int MT, int R>
__device__ __forceinline__ static void fourier_forward_body(const FourierArgs &a, const double *__restrict__ src2,
                                                            int blk) {
    extern __shared__ __align__(16) unsigned char fourier_smem[];
    constexpr int NT = kRowThreads * R;
    cplx *buf = reinterpret_cast<cplx *>(fourier_smem);
    const int M = MT > 0 ? MT : a.M, N = a.N;
    const cplx *src = reinterpret_cast<const cplx *>(src2);
    const int j0 = 1 + R * blk;
    for (int t = threadIdx.x; t < R * M; t += NT) {
        const int row = t / M, i = t - row * M, j = j0 + row;
        cplx v = {0, 0};
        if (j <= N) {
            v = src[(size_t)i + (size_t)M * j];
            const int il = i == 0 ? M - 1 : i - 1, ir = i == M - 1 ? 0 : i + 1;
            if (j == 1)
                v = less_wall(a, v, wall_node(a, src, i, 0), wall_node(a, src, il, 0), wall_node(a, src, ir, 0), 1);
            if (j == N)
                v = less_wall(a, v, wall_node(a, src, i, N + 1), wall_node(a, src, il, N + 1),
                              wall_node(a, src, ir, N + 1), -1);
        }
        buf[row * fpad(M) + fpad(i)] = v;
    }
    __syncthreads();
    store_modes<MT, R>(a, buf, j0);
}

// the same with the source formed here (shear_sim.cc:399-409, node_force)
// and written on the way, which saves reading it back: a thread runs down a
// column, so each stress is loaded once for the two rows it enters
template <int MT, int R>
__device__ __forceinline__ static void fourier_source_body(const FourierArgs &a, const SourceArgs &f,
                                                           double *__restrict__ src2, int blk) {
    extern __shared__ __align__(16) unsigned char fourier_smem[];
    constexpr int NT = kRowThreads * R;
    cplx *buf = reinterpret_cast<cplx *>(fourier_smem);
    const int M = MT > 0 ? MT : a.M, N = a.N;
    cplx *src = reinterpret_cast<cplx *>(src2);
    const int j0 = 1 + R * blk;
    const cplx low = {-f.wall, 0}, high = {f.wall, 0};
    for (int i = threadIdx.x; i < M; i += NT) {
        const int il = i == 0 ? M - 1 : i - 1;
        // cell rows j - 1 (plane row j) and j
        double p[4][R + 1], q[4][2];
#pragma unroll
        for (int row = 0; row <= R; row++) {
            const size_t o = (size_t)M * min(j0 + row, N + 1);
#pragma unroll
            for (int k = 0; k < 4; k++) p[k][row] = f.f[k][o + i];
        }
#pragma unroll
        for (int k = 0; k < 4; k++) q[k][1] = f.f[k][(size_t)M * j0 + il];
#pragma unroll
        for (int row = 0; row < R; row++) {
            const int j = j0 + row;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                q[k][0] = q[k][1];
                q[k][1] = f.f[k][(size_t)M * min(j + 1, N + 1) + il];
            }
            cplx v = {0, 0};
            if (j <= N) {
                node_force(q[0][0], p[0][row], q[0][1], p[0][row + 1], q[1][0], p[1][row], q[1][1], p[1][row + 1],
                           q[2][0], p[2][row], q[2][1], p[2][row + 1], q[3][0], p[3][row], q[3][1], p[3][row + 1],
                           f.xfac, f.yfac, v.x, v.y);
                src[(size_t)i + (size_t)M * j] = v;
                if (j == 1) {
                    const cplx w = {a.wix * low.x, a.wiy * low.y};
                    v = less_wall(a, v, w, w, w, 1);
                }
                if (j == N) {
                    const cplx w = {a.wix * high.x, a.wiy * high.y};
                    v = less_wall(a, v, w, w, w, -1);
                }
            }
            buf[row * fpad(M) + fpad(i)] = v;
        }
        if (blk == 0) {
            src[i] = low;
            src[(size_t)i + (size_t)M * (N + 1)] = high;
        }
    }
    __syncthreads();
    store_modes<MT, R>(a, buf, j0);
}

// inverse launch body: the modes of R interior rows back to (u, v),
// stored (or added); the first workgroup also writes the wall rows
template <int MT, int R>
__device__ __forceinline__ static void fourier_inverse_body(const FourierArgs &a, const double *__restrict__ src2,
                                                            double *__restrict__ z2, bool add, int blk) {
    constexpr int NT = kRowThreads * R;
    extern __shared__ __align__(16) unsigned char fourier_smem[];
    cplx *buf = reinterpret_cast<cplx *>(fourier_smem);
    const int M = MT > 0 ? MT : a.M, N = a.N, K = M / 2 + 1;
    const int j0 = 1 + R * blk;
    const double2 *S = reinterpret_cast<const double2 *>(a.S);
    cplx *z = reinterpret_cast<cplx *>(z2);
    // conjugates of the modes of u + i v, so that the forward transform is
    // the conjugate of the inverse one
    for (int t = threadIdx.x; t < R * K; t += NT) {
        const int row = t % R, k = t / R, j = j0 - 1 + row;
        double2 u = make_double2(0, 0), w = u;
        if (j < N) {
            const double2 *s = S + 2 * ((size_t)k * a.NP + j);
            u = s[0];
            w = s[1];
        }
        buf[row * fpad(M) + fpad(k)] = {u.x - w.x, w.y - u.y};
        if (k > 0 && 2 * k < M) buf[row * fpad(M) + fpad(M - k)] = {u.x + w.x, u.y + w.y};
    }
    __syncthreads();
    const cplx *c = transform_rows<MT, R>(a, buf);
    const double sc = 0.5 / M;
    for (int t = threadIdx.x; t < R * M; t += NT) {
        const int row = t / M, i = t - row * M, j = j0 + row;
        if (j > N) continue;
        const cplx v = c[row * fpad(M) + fpad(i)];
        cplx *o = z + (size_t)i + (size_t)M * j;
        if (add) *o = {fmav(sc, v.x, o->x), fmav(-sc, v.y, o->y)};
        else *o = {sc * v.x, -sc * v.y};
    }
    if (blk == 0) {
        const cplx *src = reinterpret_cast<const cplx *>(src2);
        for (int t = threadIdx.x; t < 2 * M; t += NT) {
            const int i = t % M, j = t < M ? 0 : N + 1;
            const cplx w = wall_node(a, src, i, j);
            cplx *o = z + (size_t)i + (size_t)M * j;
            if (add) *o = *o + w;
            else *o = w;
        }
    }
}

// ---------------------------------------------------------------------------
// the mode solve
// ---------------------------------------------------------------------------
// per-mode table: F, D^{-1}, -P (I + G P)^{-1}, then F^P 2^s for s = 0..6
// (row-major 2x2 blocks)
constexpr int kModePow = 7;
constexpr int kModeTab = 4 * (3 + kModePow);

// (u, v') of a row: its real or its imaginary part.  The two are solved by
// waves of their own (the blocks are real), which halves the registers and
// lane exchanges of each and doubles the waves in flight.
struct v2 { double u, w; };

// r += A x with A row-major 2x2 acting on (u, v')
__device__ __forceinline__ static void mad2(const double *A, const v2 &x, v2 &r) {
    r.u = fmav(A[1], x.w, fmav(A[0], x.u, r.u));
    r.w = fmav(A[3], x.w, fmav(A[2], x.u, r.w));
}
__device__ __forceinline__ static void mad2t(const double *A, const v2 &x, v2 &r) {  // transpose
    r.u = fmav(A[2], x.w, fmav(A[0], x.u, r.u));
    r.w = fmav(A[3], x.w, fmav(A[1], x.u, r.w));
}
__device__ __forceinline__ static v2 mul2(const double *A, const v2 &x) {
    v2 r = {0, 0};
    mad2(A, x, r);
    return r;
}
template <bool UP> __device__ __forceinline__ static v2 lane_shift(const v2 &x, int d) {
    // the value d lanes below (UP) or above; zero past the wave's end
    const int lane = threadIdx.x & 63;
    v2 r;
    if (UP) {
        r = {__shfl_up(x.u, d, 64), __shfl_up(x.w, d, 64)};
        if (lane < d) r = {0, 0};
    } else {
        r = {__shfl_down(x.u, d, 64), __shfl_down(x.w, d, 64)};
        if (lane + d >= 64) r = {0, 0};
    }
    return r;
}

// carry into each lane of a recurrence whose lanes' own results are `t`:
// the inclusive scan of t with the factor F^P per lane (or its transpose,
// backwards), shifted by one lane; the W waves of a part combined through
// `xw` in LDS (`wave`: this one of them)
template <int W, bool UP>
__device__ __forceinline__ static v2 scan_carry(const double *pw, v2 t, v2 *xw, int wave) {
#pragma unroll
    for (int s = 0; s < 6; s++) {
        const v2 n = lane_shift<UP>(t, 1 << s);
        if (UP) mad2(pw + 4 * s, n, t);
        else mad2t(pw + 4 * s, n, t);
    }
    v2 c = lane_shift<UP>(t, 1);
    if constexpr (W > 1) {
        const int lane = threadIdx.x & 63;
        __syncthreads();
        if (lane == (UP ? 63 : 0)) xw[wave] = t;
        __syncthreads();
        // the waves before (after) this one, combined in their order
        v2 in = {0, 0};
#pragma unroll
        for (int q = 0; q < W - 1; q++) {
            const int w = UP ? q : W - 1 - q;
            if (UP ? w < wave : w > wave) {
                v2 r = xw[w];
                if (UP) mad2(pw + 4 * 6, in, r);
                else mad2t(pw + 4 * 6, in, r);
                in = r;
            }
        }
        // times F^{P lane}: the powers of this lane's bits
        const int d = UP ? lane : 63 - lane;
#pragma unroll
        for (int s = 0; s < 6; s++)
            if ((d >> s) & 1) {
                v2 r = {0, 0};
                if (UP) mad2(pw + 4 * s, in, r);
                else mad2t(pw + 4 * s, in, r);
                in = r;
            }
        c = {c.u + in.u, c.w + in.w};
    }
    return c;
}

// LDS column of a mode: row j of P rows per thread at slot 2 j + (j / P), in
// 16-byte units (u complex, v' complex): a thread's rows are contiguous and
// threads start one slot apart in the banks
template <int P> __host__ __device__ constexpr int mode_slot(int j) { return 2 * j + j / P; }

template <int W, int P>
__device__ __forceinline__ static void fourier_mode_body(const FourierArgs &a, int k) {
    extern __shared__ __align__(16) unsigned char fourier_smem[];
    constexpr int NT = 128 * W;
    double2 *col = reinterpret_cast<double2 *>(fourier_smem);
    __shared__ v2 xw[2][W];
    __shared__ v2 first[2];
    const int N = a.N, tid = threadIdx.x;
    const int part = tid / (64 * W), ln = tid % (64 * W);  // real or imaginary part; lane of it
    const int wave = ln >> 6;
    const double *tab = a.tab + (size_t)kModeTab * k;
    const double *F = tab, *Di = tab + 4, *C = tab + 8, *pw = tab + 12;
    double2 *S = reinterpret_cast<double2 *>(a.S) + (size_t)2 * k * a.NP;
    // the column, coalesced, all of a thread's loads in flight
    double2 in[P];
#pragma unroll
    for (int q = 0; q < P; q++) {
        const int t = tid + NT * q;
        in[q] = S[t < 2 * N ? t : 0];
    }
#pragma unroll
    for (int q = 0; q < P; q++) {
        const int t = tid + NT * q;
        col[mode_slot<P>(t >> 1) + (t & 1)] = t < 2 * N ? in[q] : make_double2(0, 0);
    }
    __syncthreads();
    v2 g[P];
    const int r0 = ln * P;
    // this part of the thread's rows (u at even, v' at odd places)
    double *mine = reinterpret_cast<double *>(col + mode_slot<P>(r0)) + part;
#pragma unroll
    for (int p = 0; p < P; p++) g[p] = {mine[4 * p], mine[4 * p + 2]};
    // forward: g_j = f_j + F g_{j-1}
#pragma unroll
    for (int p = 1; p < P; p++) mad2(F, g[p - 1], g[p]);
    v2 c = scan_carry<W, true>(pw, g[P - 1], xw[part], wave);
#pragma unroll
    for (int p = 0; p < P; p++) {
        c = mul2(F, c);
        g[p] = {g[p].u + c.u, g[p].w + c.w};
        if (r0 + p >= N) g[p] = {0, 0};
    }
    // backward for the first row only: y_1
    v2 y = mul2(Di, g[P - 1]);
#pragma unroll
    for (int p = P - 2; p >= 0; p--) {
        v2 t = mul2(Di, g[p]);
        mad2t(F, y, t);
        y = t;
    }
    v2 t0 = scan_carry<W, false>(pw, y, xw[part], wave);
    if (ln == 0) {
        // y_1 = this thread's own part + E^P times the carry from the next
        mad2t(pw, t0, y);
        first[part] = mul2(C, y);  // -P w_1
    }
    __syncthreads();
    // g_j += F^{j-1} (-P w_1)
    v2 h = first[part];
#pragma unroll
    for (int s = 0; s < 6; s++)
        if ((ln >> s) & 1) h = mul2(pw + 4 * s, h);
    if constexpr (W > 1)
        for (int w = 0; w < wave; w++) h = mul2(pw + 4 * 6, h);
#pragma unroll
    for (int p = 0; p < P; p++) {
        if (r0 + p < N) g[p] = {g[p].u + h.u, g[p].w + h.w};
        h = mul2(F, h);
    }
    // backward: w_j = D^{-1} g_j + E w_{j+1}
    g[P - 1] = mul2(Di, g[P - 1]);
#pragma unroll
    for (int p = P - 2; p >= 0; p--) {
        v2 t = mul2(Di, g[p]);
        mad2t(F, g[p + 1], t);
        g[p] = t;
    }
    c = scan_carry<W, false>(pw, g[0], xw[part], wave);
#pragma unroll
    for (int p = P - 1; p >= 0; p--) {
        v2 t = {0, 0};
        mad2t(F, c, t);
        c = t;
        mine[4 * p] = g[p].u + c.u;
        mine[4 * p + 2] = g[p].w + c.w;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < P; q++) {
        const int t = tid + NT * q;
        if (t < 2 * N) S[t] = col[mode_slot<P>(t >> 1) + (t & 1)];
    }
}

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
template <int MT, int R>
__global__ void __launch_bounds__(kRowThreads *R) fourier_forward_kernel(FourierArgs a, const double *src) {
    fourier_forward_body<MT, R>(a, src, blockIdx.x);
}
template <int MT, int R>
__global__ void __launch_bounds__(kRowThreads *R) fourier_source_kernel(FourierArgs a, SourceArgs f, double *src) {
    fourier_source_body<MT, R>(a, f, src, blockIdx.x);
}
template <int MT, int R>
__global__ void __launch_bounds__(kRowThreads *R) fourier_inverse_kernel(FourierArgs a, const double *src, double *z,
                                                                         bool add) {
    fourier_inverse_body<MT, R>(a, src, z, add, blockIdx.x);
}
template <int W, int P> __global__ void __launch_bounds__(128 * W) fourier_mode_kernel(FourierArgs a) {
    fourier_mode_body<W, P>(a, blockIdx.x);
}

// the same over the members of an ensemble (batch.h) that solve this way;
// members whose slot flag is clear return at once, and those past their first
// test solve for the residual and add
template <int MT>
__global__ void __launch_bounds__(2 * kRowThreads) fourier_forward_batch_kernel(const FourierEntry *E, const int *map,
                                                                                const EnsState *St) {
    const int2 el = batch_slot(map, blockIdx.x);
    const FourierEntry &x = E[el.x];
    if (!St[x.member].active) return;
    const FourierArgs a = x.a;
    fourier_forward_body<MT, 2>(a, St[x.member].phase == ENS_LOOP ? x.r : x.src, el.y);
}
template <int MT>
__global__ void __launch_bounds__(2 * kRowThreads) fourier_inverse_batch_kernel(const FourierEntry *E, const int *map,
                                                                                const EnsState *St) {
    const int2 el = batch_slot(map, blockIdx.x);
    const FourierEntry &x = E[el.x];
    if (!St[x.member].active) return;
    const FourierArgs a = x.a;
    const bool add = St[x.member].phase == ENS_LOOP;
    fourier_inverse_body<MT, 2>(a, add ? x.r : x.src, x.z, add, el.y);
}
template <int W, int P>
__global__ void __launch_bounds__(128 * W) fourier_mode_batch_kernel(const FourierEntry *E, const int *map,
                                                                     const EnsState *St) {
    const int2 el = batch_slot(map, blockIdx.x);
    const FourierEntry &x = E[el.x];
    if (!St[x.member].active) return;
    const FourierArgs a = x.a;
    fourier_mode_body<W, P>(a, el.y);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// lengths with the in-place transform of compile-time length
static bool fixed_length(int M) { return M == 128 || M == 256 || M == 512 || M == 1024 || M == 2048 || M == 4096; }

// rows per workgroup of a grid's own launches
static int row_group(int M, int N) { return fixed_length(M) && M >= 512 && M <= 2048 && N >= 4 * 255 ? 4 : 2; }
// the largest prime factor from 7 on (0: none)
static int large_prime(int M) {
    for (int r : {2, 3, 5})
        while (M % r == 0) M /= r;
    int big = M > 1 ? M : 0;
    for (int r = 7; M > 1; r += 2)
        for (; M % r == 0; M /= r) big = r;
    return big;
}
// the rows (twice for a transform that is not in place) and a prime's roots
static size_t row_lds(int M, int R) {
    if (fixed_length(M)) return (size_t)R * fpad(M) * sizeof(cplx);
    return (size_t)(2 * R * fpad(M) + large_prime(M)) * sizeof(cplx);
}
size_t fourier_row_lds(int M) { return row_lds(M, 2); }
// the most a row launch of any length takes (fourier_fits)
constexpr size_t kMaxRowLds = 152 * 1024;

// rows per thread and waves per part of a mode: eight rows a thread, fewer
// where one wave then covers the column
static int mode_rows(int N) { return N <= 128 ? 2 : (N <= 256 ? 4 : 8); }
static int mode_waves(int N) { return N <= 512 ? 1 : (N <= 1024 ? 2 : (N <= 2048 ? 4 : 8)); }
size_t fourier_mode_lds(int N) {
    const int rows = 64 * mode_waves(N) * mode_rows(N);
    return (size_t)(2 * rows + rows / mode_rows(N)) * 16;
}

bool fourier_fits(int M, int n) {
    const int N = n - 2;  // n node rows, walls included
    return M >= 4 && M <= 4096 && N >= 1 && N <= 4096 && fourier_row_lds(M) <= kMaxRowLds;
}

// f(integral_constant) of the row kernels' compile-time length (0: any)
template <typename F> static int with_length(int M, F f) {
    switch (fixed_length(M) ? M : 0) {
    case 128: return f(std::integral_constant<int, 128>());
    case 256: return f(std::integral_constant<int, 256>());
    case 512: return f(std::integral_constant<int, 512>());
    case 1024: return f(std::integral_constant<int, 1024>());
    case 2048: return f(std::integral_constant<int, 2048>());
    case 4096: return f(std::integral_constant<int, 4096>());
    default: return f(std::integral_constant<int, 0>());
    }
}
// f(waves, rows per thread) of the mode kernel for N interior rows
template <typename F> static int with_column(int N, F f) {
    typedef std::integral_constant<int, 8> eight;
    const int W = mode_waves(N), P = mode_rows(N);
    if (W == 1 && P == 2) return f(std::integral_constant<int, 1>(), std::integral_constant<int, 2>());
    if (W == 1 && P == 4) return f(std::integral_constant<int, 1>(), std::integral_constant<int, 4>());
    if (W == 1) return f(std::integral_constant<int, 1>(), eight());
    if (W == 2) return f(std::integral_constant<int, 2>(), eight());
    if (W == 4) return f(std::integral_constant<int, 4>(), eight());
    return f(eight(), eight());
}

template <typename K> static int allow_lds(K kernel, size_t bytes) {
    if (bytes <= 64 * 1024) return STZ_OK;
    STZ_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)bytes));
    return STZ_OK;
}

// f(integral_constant) of the rows per workgroup of a grid's own launches:
// four only with the lengths row_group gives them to
template <int MT, typename F> static int with_rows(int M, int N, F f) {
    if constexpr (MT >= 512 && MT <= 2048)
        if (row_group(M, N) == 4) return f(std::integral_constant<int, 4>());
    return f(std::integral_constant<int, 2>());
}

// Raise the LDS limit of the kernels a grid uses (once per operator set-up).
// The limit belongs to the kernel, not to a grid: a kernel of one length or
// one column variant always takes the same, the general-length ones get the
// most that any length takes, so that no grid lowers it for another.
int fourier_set_lds_limit(const FourierArgs &a) {
    const size_t ml = fourier_mode_lds(a.N);
    const int e = with_length(a.M, [&](auto mt) {
        constexpr int MT = decltype(mt)::value;
        const size_t bl = MT > 0 ? fourier_row_lds(a.M) : kMaxRowLds;
        int r;
        if ((r = allow_lds(fourier_forward_batch_kernel<MT>, bl)) ||
            (r = allow_lds(fourier_inverse_batch_kernel<MT>, bl)))
            return r;
        return with_rows<MT>(a.M, a.N, [&](auto rr) {
            constexpr int R = decltype(rr)::value;
            const size_t rl = MT > 0 ? row_lds(a.M, R) : kMaxRowLds;
            int q;
            if ((q = allow_lds(fourier_forward_kernel<MT, R>, rl)) || (q = allow_lds(fourier_source_kernel<MT, R>, rl)))
                return q;
            return allow_lds(fourier_inverse_kernel<MT, R>, rl);
        });
    });
    if (e) return e;
    return with_column(a.N, [&](auto w, auto p) {
        constexpr int W = decltype(w)::value, P = decltype(p)::value;
        const int r = allow_lds(fourier_mode_kernel<W, P>, ml);
        return r ? r : allow_lds(fourier_mode_batch_kernel<W, P>, ml);
    });
}

int fourier_row_workgroups(int N) { return (N + 1) / 2; }
int fourier_row_variant(int M) { return fixed_length(M) ? M : 0; }
int fourier_mode_variant(int N) { return 16 * mode_waves(N) + mode_rows(N); }

// z = A^{-1} src, or (add) z += A^{-1} src; with f the source is formed first
int mg_fourier_solve(const FourierArgs &a, const SourceArgs *f, double *src, double *z, bool add, hipStream_t st) {
    const size_t ml = fourier_mode_lds(a.N);
    auto rows = [&](auto launch) {
        with_length(a.M, [&](auto mt) {
            constexpr int MT = decltype(mt)::value;
            return with_rows<MT>(a.M, a.N, [&](auto rr) {
                constexpr int R = decltype(rr)::value;
                launch(mt, rr, dim3((a.N + R - 1) / R), dim3(kRowThreads * R), row_lds(a.M, R));
                return 0;
            });
        });
    };
    rows([&](auto mt, auto rr, dim3 g, dim3 b, size_t lds) {
        constexpr int MT = decltype(mt)::value, R = decltype(rr)::value;
        if (f) hipLaunchKernelGGL((fourier_source_kernel<MT, R>), g, b, lds, st, a, *f, src);
        else hipLaunchKernelGGL((fourier_forward_kernel<MT, R>), g, b, lds, st, a, (const double *)src);
    });
    with_column(a.N, [&](auto w, auto p) {
        constexpr int W = decltype(w)::value, P = decltype(p)::value;
        hipLaunchKernelGGL((fourier_mode_kernel<W, P>), dim3(a.M / 2 + 1), dim3(128 * W), ml, st, a);
        return 0;
    });
    rows([&](auto mt, auto rr, dim3 g, dim3 b, size_t lds) {
        constexpr int MT = decltype(mt)::value, R = decltype(rr)::value;
        hipLaunchKernelGGL((fourier_inverse_kernel<MT, R>), g, b, lds, st, a, (const double *)src, z, add);
    });
    STZ_HIP(hipGetLastError());
    return STZ_OK;
}

int batch_fourier_rows(bool inverse, int M, size_t lds, const FourierEntry *E, const int *map, int total,
                       const EnsState *St, hipStream_t st) {
    if (total == 0) return STZ_OK;
    with_length(M, [&](auto mt) {
        constexpr int MT = decltype(mt)::value;
        if (inverse)
            hipLaunchKernelGGL((fourier_inverse_batch_kernel<MT>), dim3(total), dim3(2 * kRowThreads), lds, st, E, map, St);
        else
            hipLaunchKernelGGL((fourier_forward_batch_kernel<MT>), dim3(total), dim3(2 * kRowThreads), lds, st, E, map, St);
        return 0;
    });
    STZ_HIP(hipGetLastError());
    return STZ_OK;
}

int batch_fourier_modes(int N, const FourierEntry *E, const int *map, int total, const EnsState *St,
                        hipStream_t st) {
    if (total == 0) return STZ_OK;
    const size_t ml = fourier_mode_lds(N);
    with_column(N, [&](auto w, auto p) {
        constexpr int W = decltype(w)::value, P = decltype(p)::value;
        hipLaunchKernelGGL((fourier_mode_batch_kernel<W, P>), dim3(total), dim3(128 * W), ml, st, E, map, St);
        return 0;
    });
    STZ_HIP(hipGetLastError());
    return STZ_OK;
}

// ---------------------------------------------------------------------------
// host set-up
// ---------------------------------------------------------------------------
namespace {
typedef long double real;
struct m2 { real a, b, c, d; };
m2 operator*(const m2 &x, const m2 &y) {
    return {x.a * y.a + x.b * y.c, x.a * y.b + x.b * y.d, x.c * y.a + x.d * y.c, x.c * y.b + x.d * y.d};
}
m2 operator+(const m2 &x, const m2 &y) { return {x.a + y.a, x.b + y.b, x.c + y.c, x.d + y.d}; }
m2 operator-(const m2 &x, const m2 &y) { return {x.a - y.a, x.b - y.b, x.c - y.c, x.d - y.d}; }
m2 neg(const m2 &x) { return {-x.a, -x.b, -x.c, -x.d}; }
m2 tr(const m2 &x) { return {x.a, x.c, x.b, x.d}; }
m2 inv(const m2 &x) {
    const real r = 1 / (x.a * x.d - x.b * x.c);
    return {x.d * r, -x.b * r, -x.c * r, x.a * r};
}
real big(const m2 &x) { return std::fmax(std::fmax(std::fabs(x.a), std::fabs(x.b)), std::fmax(std::fabs(x.c), std::fabs(x.d))); }
}  // namespace

size_t fourier_spectrum_elems(int M, int N) { return (size_t)4 * (M / 2 + 1) * ((N + 3) & ~3); }
static size_t table_elems(int M) { return (size_t)4 * M + (size_t)kModeTab * (M / 2 + 1); }

// The constants of the solve for M x (N + 2) nodes with the interior stencil
// s40 and the wall rows' stencil w40 (sim.hip, top_row_stencil): T receives
// the stages' twiddles, the M roots of unity e^{-2 pi i m / M} and, from element
// 4 M on, the mode tables.  Returns false
// if the operator does not have the form above or a mode is singular.
bool fourier_setup(const double *s40, const double *w40, int M, int N, FourierArgs &a, std::vector<double> &T) {
    a.M = M;
    a.N = N;
    a.NP = (N + 3) & ~3;
    a.nst = 0;
    int left = M;
    if (fixed_length(M))
        while (left > 1) {
            a.radix[a.nst++] = fixed_radix(left);
            left /= fixed_radix(left);
        }
    // the primes first: the first stage has no twiddles
    for (int big = large_prime(left); big >= 7; big = large_prime(left)) {
        a.radix[a.nst++] = big;
        left /= big;
    }
    for (int r : {8, 4, 2, 3, 5})
        while (left % r == 0) {
            a.radix[a.nst++] = r;
            left /= r;
        }
    // the pattern of qs_multi's operator: edges diagonal, corners +-q off the
    // diagonal, walls diagonal
    const real xx = s40[12], xy = s40[15], yx = s40[4], yy = s40[7], q = s40[1];
    if (!sparse_pattern(s40) || s40[20] != s40[12] || s40[23] != s40[15] || s40[28] != s40[4] ||
        s40[31] != s40[7] || s40[2] != s40[1] || s40[9] != -s40[1] || s40[10] != -s40[1] || s40[25] != -s40[1] ||
        s40[26] != -s40[1] || s40[33] != s40[1] || s40[34] != s40[1])
        return false;
    for (int k = 0; k < 36; k++)
        if (w40[k] != 0 && k != 16 && k != 19) return false;
    a.cxx = s40[4];
    a.cyy = s40[7];
    a.cxy = s40[1];
    a.wix = w40[36];
    a.wiy = w40[39];
    T.assign(table_elems(M), 0.0);
    const real pi = 3.14159265358979323846264338327950288L;
    double *root = T.data() + 2 * (size_t)M;
    for (int m = 0; m < M; m++) {
        const real th = 2 * pi * m / M;
        root[2 * m] = (double)std::cos(th);
        root[2 * m + 1] = (double)-std::sin(th);
    }
    // the stage after a product of L: entries (q - 1) L + k from L - 1 on
    for (int s = 0, L = 1; s < a.nst; L *= a.radix[s++])
        for (int q = 1; q < a.radix[s]; q++)
            for (int k = 0; k < L; k++) {
                const size_t o = (size_t)(L - 1) + (size_t)(q - 1) * L + k, r = (size_t)k * q * (M / (L * a.radix[s]));
                T[2 * o] = root[2 * r];
                T[2 * o + 1] = root[2 * r + 1];
            }
    const int P = mode_rows(N);
    const real e0 = (real)s40[16] + 2 * xx + 2 * yx, e1 = (real)s40[19] + 2 * xy + 2 * yy;  // row sums: rounding
    for (int k = 0; k <= M / 2; k++) {
        const real th = pi * k / M, sh = std::sin(th) * std::sin(th);
        const real sn = 2 * k == M ? 0 : 2 * q * std::sin(2 * th);
        // cc + 2 cos(theta) edge = (row sum) - 2 edge_y - 4 sin^2(theta/2) edge_x;
        // the row sum is zero but for rounding, which the residual keeps
        const m2 B = {e0 - 2 * yx - 4 * sh * xx, 0, 0, e1 - 2 * yy - 4 * sh * xy};
        const m2 Cu = {yx, -sn, sn, yy}, Cd = tr(Cu);
        m2 D;
        if (k == 0) {
            D = {-yx, 0, 0, -yy};
        } else {
            m2 b = B, u = Cu, d = Cd;
            D = B;
            for (int it = 0; it < 64; it++) {
                const m2 s = inv(b), us = u * s, ds = d * s, step = ds * u;
                D = D - step;
                b = b - us * d - step;
                u = neg(us * u);
                d = neg(ds * d);
                if (big(step) <= 1e-22L * big(D)) break;
            }
        }
        const m2 Di = inv(D), F = neg(Cd * Di);
        // G = (M^{-1})_11 = sum_{m < N} (F^T)^m D^{-1} F^m, by doubling over N's bits
        m2 G = Di, Fn = F;
        int bit = 0;
        while ((2 << bit) <= N) bit++;
        for (bit--; bit >= 0; bit--) {
            G = G + tr(Fn) * G * Fn;
            Fn = Fn * Fn;
            if ((N >> bit) & 1) {
                G = Di + tr(F) * G * F;
                Fn = Fn * F;
            }
        }
        // P keeps the row-sum rounding out (mode 0: P = -Cu exactly)
        const m2 Pm = k == 0 ? m2{-yx, 0, 0, -yy} : B - D;
        const m2 one = {1, 0, 0, 1};
        const m2 Cm = neg(Pm * inv(one + G * Pm));
        double *t = T.data() + 4 * (size_t)M + (size_t)kModeTab * k;
        auto put = [](double *o, const m2 &x) {
            o[0] = (double)x.a;
            o[1] = (double)x.b;
            o[2] = (double)x.c;
            o[3] = (double)x.d;
        };
        put(t, F);
        put(t + 4, Di);
        put(t + 8, Cm);
        m2 Fp = F;
        for (int p = 1; p < P; p++) Fp = Fp * F;
        for (int s = 0; s < kModePow; s++) {
            put(t + 12 + 4 * s, Fp);
            Fp = Fp * Fp;
        }
        for (int r = 0; r < kModeTab; r++)
            if (!std::isfinite(t[r])) return false;
    }
    return true;
}

}  // namespace stz
