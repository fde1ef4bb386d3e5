// DCT and DST of types 1-4 over any set of axes, FP64, with the semantics of
// pocketfft::dct / pocketfft::dst (pocketfft_hdronly.h:3284-3318): unnormalised
// sums, `ortho` applying only the end-point scalings the reference applies
// (the overall 1/sqrt factor is the caller's fct), fct on the first axis.
//
// Each axis of length N runs one c2c transform per line through the engine's
// own FP64 plan over a workspace, between a pre-pass that builds the complex
// sequence from the strided input and a post-pass that forms the outputs.
//
// Types 2-4 at even N (M = N/2 points per line, after Makhoul): with x' the
// input as the DCT sees it -- x'[n] = (-1)^n x[n] for DST-II, x'[n] = x[N-1-n]
// for DST-III / DST-IV (DST-II(x)[k] = DCT-II(x')[N-1-k], DST-III(x)[k] =
// (-1)^k DCT-III(x')[k], DST-IV(x)[k] = (-1)^k DCT-IV(x')[k]) --
//   DCT-II   z[p] = v[2p] + i v[2p+1], v[q] = x'[2q] (q < M), x'[2N-2q-1] (q >= M)
//            forward; V[k] = E[k] + e^{-2 pi i k/N} O[k] from Z[k], conj Z[M-k];
//            W = e^{-i pi k/2N} V[k]; y[k] = 2 Re W, y[N-k] = -2 Im W (k = 0..M)
//   DCT-III  V(k) = e^{i pi k/2N} (x'[k] - i x'[N-k]) (x'[N] = 0), k = 0..M;
//            z[k] = (V(k) + conj V(M-k)) + i e^{2 pi i k/N} (V(k) - conj V(M-k));
//            backward; v[2n] = Re Z[n], v[2n+1] = Im Z[n]; y[2q] = v[q],
//            y[2q+1] = v[N-1-q]
//   DCT-IV   z[p] = (x'[2p] + i x'[N-1-2p]) e^{-i pi p/N}; forward;
//            S = e^{-i pi (4k+1)/4N} Z[k]; y[2k] = 2 Re S, y[N-1-2k] = -2 Im S
// Types 1 and odd N (L points per line):
//   DCT-I    z = even extension of x, L = 2(N-1)  forward   y[k] = Re Z[k]
//   DST-I    z = (0, x, 0, -x~), L = 2(N+1)       forward   y[k] = -Im Z[k+1]
//   DCT-II   z = x, zero-padded, L = 2N           forward   y[k] = 2 Re(e^{-i pi k/2N} Z[k])
//   DST-II   z = x, zero-padded                   forward   y[k] = -2 Im(e^{-i pi (k+1)/2N} Z[k+1])
//   DCT-III  z[n] = x''[n] e^{i pi n/2N}, x''[0] = x[0], x''[n] = 2 x[n]
//                                                 backward  y[k] = Re c[k]
//   DST-III  z[m] = x''[m] e^{i pi m/2N}, m = 1..N, x''[m] = 2 x[m-1] (m < N), x''[N] = x[N-1]
//                                                 backward  y[k] = Im c[k]
//   DCT-IV   z[n] = x[n] e^{-i pi (2n+1)/4N}      forward   y[k] = 2 Re(e^{-i pi k/2N} Z[k])
//   DST-IV   as DCT-IV                            forward   y[k] = -2 Im(e^{-i pi k/2N} Z[k])
// (each follows from writing the cosine / sine as the real / imaginary part of
// one exponential and collecting the DFT kernel).  The half-length forms take
// their pre / post twiddles, and the one-kernel path its stage twiddles, from
// per-axis tables written by the long-double host generator (one length per
// axis, so one table serves every line); the full-length forms use FP64
// sincospi.
//
// Workspace layout per axis: [lines, L] when the axis is the input's unit-
// stride dimension (threads walk along a line), else [L, lines] (threads walk
// across lines, which keeps the strided gathers and scatters coalesced; the
// c2c then runs over the workspace's strided axis).
#include <cmath>
#include <type_traits>
#include <vector>

#include "butterflies.h"
#include "engine.h"
#include "line_reach.h"
#include "mix_fft.h"

namespace ifft {

constexpr int kMaxDims = kMaxBatchDims + 1;
static_assert(kMaxDims == kLineDims, "a LineMap holds every dimension");

struct R2rParams {
    const double *src;
    double *dst;
    double2 *work;
    LineMap in, out;
    long long sa_in, sa_out;   // element stride along the axis
    long long N, L, lines;
    int cosine, type, ortho;
    int half;                  // types 2-4 at even N: L = N/2 points per line
    int col;                   // workspace [L, lines] (line fastest) instead of [lines, L]
    double fct;
    // half-length lines: the twiddles of the pre / post steps, L + 1 entries each
    // (types 2, 3: e1[k] = exp(i pi 2k / N), e2[k] = exp(i pi k / 2N);
    //  type 4: e1[k] = exp(i pi k / N), e2[k] = exp(i pi (4k + 1) / 4N))
    const double2 *e1, *e2;
};

// (line, point) of work item e and the workspace index of that point
__device__ __forceinline__ void r2r_item(const R2rParams &P, long long e, long long cnt, long long &line, long long &m)
{
    if (P.col) {
        m = e / P.lines;
        line = e - m * P.lines;
    } else {
        line = e / cnt;
        m = e - line * cnt;
    }
}

__device__ __forceinline__ long long r2r_widx(const R2rParams &P, long long line, long long m)
{
    return P.col ? m * P.lines + line : line * P.L + m;
}

__device__ __forceinline__ long long line_off(const LineMap &m, long long line)
{
    long long off = 0;
    for (int d = m.nd - 1; d >= 0; --d) {
        const long long c = m.cnt[d];
        off += (line % c) * m.st[d];
        line /= c;
    }
    return off;
}

// exp(i pi a / b)
__device__ __forceinline__ double2 expipi(double a, double b)
{
    double s, c;
    sincospi(a / b, &s, &c);
    return make_double2(c, s);
}

constexpr double kSqrt2 = 1.4142135623730951;

// input point n as the half-length DCT sees it (DST sign / reversal, type-3 ortho)
template <int TYPE>
__device__ __forceinline__ double r2r_xp(const R2rParams &P, const double *x, long long n)
{
    const long long N = P.N;
    const long long orig = (!P.cosine && TYPE != 2) ? N - 1 - n : n;
    double v = x[orig * P.sa_in];
    if (TYPE == 3 && P.ortho && orig == 0) v *= kSqrt2;
    if (!P.cosine && TYPE == 2 && (n & 1)) v = -v;
    return v;
}

// point m of the half-length complex sequence of one line (types 2-4, even N)
template <int TYPE>
__device__ __forceinline__ double2 half_pre(const R2rParams &P, const double *x, long long m)
{
    const long long N = P.N, M = P.L;
    if constexpr (TYPE == 2) {
        auto v = [&](long long q) {
            return q < M ? r2r_xp<2>(P, x, 2 * q) : r2r_xp<2>(P, x, 2 * N - 2 * q - 1);
        };
        return make_double2(v(2 * m), v(2 * m + 1));
    } else if constexpr (TYPE == 3) {
        auto xe = [&](long long k) { return k < N ? r2r_xp<3>(P, x, k) : 0.0; };
        auto V = [&](long long k) { return cmul(P.e2[k], make_double2(xe(k), -xe(N - k))); };
        const double2 vk = V(m), vm = cconj(V(M - m));
        const double2 sum = cadd(vk, vm);
        const double2 dif = cmul(P.e1[m], csub(vk, vm));
        return make_double2(sum.x - dif.y, sum.y + dif.x);
    } else {
        return cmul(make_double2(r2r_xp<4>(P, x, 2 * m), r2r_xp<4>(P, x, N - 1 - 2 * m)), cconj(P.e1[m]));
    }
}

__global__ void k_r2r_pre(const R2rParams P)
{
    const long long total = P.lines * P.L, N = P.N, L = P.L;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        long long line, m;
        r2r_item(P, e, L, line, m);
        const double *x = P.src + line_off(P.in, line);
        auto X = [&](long long j) { return x[j * P.sa_in]; };
        double2 z = make_double2(0.0, 0.0);
        if (P.half) {
            z = P.type == 2 ? half_pre<2>(P, x, m) : P.type == 3 ? half_pre<3>(P, x, m) : half_pre<4>(P, x, m);
        } else if (P.cosine) {
            switch (P.type) {
                case 1: {
                    const long long j = m < N ? m : L - m;
                    double v = X(j);
                    if (P.ortho && (j == 0 || j == N - 1)) v *= kSqrt2;
                    z = make_double2(v, 0.0);
                    break;
                }
                case 2:
                    if (m < N) z = make_double2(X(m), 0.0);
                    break;
                case 3:
                    if (m < N) {
                        const double v = m == 0 ? X(0) * (P.ortho ? kSqrt2 : 1.0) : 2.0 * X(m);
                        z = cscale(expipi((double)m, 2.0 * N), v);
                    }
                    break;
                default:
                    if (m < N) z = cscale(cconj(expipi((double)(2 * m + 1), 4.0 * N)), X(m));
            }
        } else {
            switch (P.type) {
                case 1:
                    if (m >= 1 && m <= N) z = make_double2(X(m - 1), 0.0);
                    else if (m >= N + 2) z = make_double2(-X(L - 1 - m), 0.0);
                    break;
                case 2:
                    if (m < N) z = make_double2(X(m), 0.0);
                    break;
                case 3:
                    if (m >= 1 && m <= N) {
                        double v = m < N ? 2.0 * X(m - 1) : X(N - 1);
                        if (P.ortho && m == 1) v *= kSqrt2;   // the reference scales input x[0]
                        z = cscale(expipi((double)m, 2.0 * N), v);
                    }
                    break;
                default:
                    if (m < N) z = cscale(cconj(expipi((double)(2 * m + 1), 4.0 * N)), X(m));
            }
        }
        P.work[r2r_widx(P, line, m)] = z;
    }
}

// output i (as the DCT forms it) of a half-length line: DST reversal / signs, scale
template <int TYPE>
__device__ __forceinline__ void r2r_put(const R2rParams &P, double *y, long long i, double v)
{
    const long long N = P.N;
    long long o = i;
    if (!P.cosine) {
        if (TYPE == 2) o = N - 1 - i;
        else if (i & 1) v = -v;
    }
    y[o * P.sa_out] = v * P.fct;
}

// work items per line of the post-pass
__host__ __device__ inline long long r2r_post_count(int half, int type, long long N)
{
    return half ? (type == 2 ? N / 2 + 1 : N / 2) : N;
}

// outputs of post item k of one half-length line from its transformed points Zat(m)
template <int TYPE, typename ZAT>
__device__ __forceinline__ void half_post(const R2rParams &P, double *yl, long long k, ZAT Zat)
{
    const long long N = P.N, M = P.L;
    if constexpr (TYPE == 2) {
        const double2 zk = Zat(k == M ? 0 : k), zm = cconj(Zat(k == 0 ? 0 : M - k));
        const double2 ev = cscale(cadd(zk, zm), 0.5);
        const double2 d = csub(zk, zm);
        const double2 od = make_double2(0.5 * d.y, -0.5 * d.x);
        const double2 V = cadd(ev, cmul(cconj(P.e1[k]), od));
        const double2 W = cmul(cconj(P.e2[k]), V);
        const long long oi = P.cosine ? 0 : N - 1;   // the ortho end point as the DCT indexes it
        double lo = 2.0 * W.x;
        if (P.ortho && k == oi) lo *= 0.5 * kSqrt2;
        r2r_put<2>(P, yl, k, lo);
        if (k > 0 && k < M) {
            double hi = -2.0 * W.y;
            if (P.ortho && N - k == oi) hi *= 0.5 * kSqrt2;
            r2r_put<2>(P, yl, N - k, hi);
        }
    } else if constexpr (TYPE == 3) {
        const double2 z = Zat(k);
        auto sigma = [&](long long q) { return q < M ? 2 * q : 2 * N - 2 * q - 1; };
        r2r_put<3>(P, yl, sigma(2 * k), z.x);
        r2r_put<3>(P, yl, sigma(2 * k + 1), z.y);
    } else {
        const double2 S = cmul(Zat(k), cconj(P.e2[k]));
        r2r_put<4>(P, yl, 2 * k, 2.0 * S.x);
        r2r_put<4>(P, yl, N - 1 - 2 * k, -2.0 * S.y);
    }
}

__global__ void k_r2r_post(const R2rParams P)
{
    const long long N = P.N;
    const long long cnt = r2r_post_count(P.half, P.type, N), total = P.lines * cnt;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        long long line, k;
        r2r_item(P, e, cnt, line, k);
        double *yl = P.dst + line_off(P.out, line);
        auto Zat = [&](long long m) { return P.work[r2r_widx(P, line, m)]; };
        if (P.half) {
            if (P.type == 2) half_post<2>(P, yl, k, Zat);
            else if (P.type == 3) half_post<3>(P, yl, k, Zat);
            else half_post<4>(P, yl, k, Zat);
            continue;
        }
        double y;
        if (P.cosine) {
            switch (P.type) {
                case 1:
                    y = Zat(k).x;
                    if (P.ortho && (k == 0 || k == N - 1)) y *= 0.5 * kSqrt2;
                    break;
                case 2:
                    y = 2.0 * cmul(cconj(expipi((double)k, 2.0 * N)), Zat(k)).x;
                    if (P.ortho && k == 0) y *= 0.5 * kSqrt2;
                    break;
                case 3:
                    y = Zat(k).x;
                    break;
                default:
                    y = 2.0 * cmul(cconj(expipi((double)k, 2.0 * N)), Zat(k)).x;
            }
        } else {
            switch (P.type) {
                case 1:
                    y = -Zat(k + 1).y;
                    break;
                case 2:
                    y = -2.0 * cmul(cconj(expipi((double)(k + 1), 2.0 * N)), Zat(k + 1)).y;
                    if (P.ortho && k == 0) y *= 0.5 * kSqrt2;
                    break;
                case 3:
                    y = Zat(k).y;
                    break;
                default:
                    y = -2.0 * cmul(cconj(expipi((double)k, 2.0 * N)), Zat(k)).y;
            }
        }
        yl[k * P.sa_out] = y * P.fct;
    }
}

// ---------------------------------------------------------------------------
// types 2-4 at even N in one kernel per axis
// ---------------------------------------------------------------------------

// A workgroup takes `tb` lines along or across which its lanes walk (col), builds each line's
// N/2-point sequence in an LDS row, runs the mixed-radix stages (mix_fft.h) there and forms the
// outputs from the row, so HBM sees each line read once and written once whatever its stride.
// The half-length forms are symmetric in (k, M - k): one pair of points shares its inputs, roots and
// products, and along a unit-stride line the real words move in aligned pairs.
//
// Measured on one MI355X (DCT-II unless said, one axis, one launch):
//   2160 x 3840 columns  0.189 -> 0.056 ms (three passes before: build, c2c, form), DCT-III 0.187 -> 0.054
//   2160 x 3840 rows     0.053 -> 0.042 ms (3.2 TB/s), DCT-III 0.072 -> 0.037
//   4096 x 4096 rows     0.078 -> 0.068 ms, columns 0.237 -> 0.115
//   8 x 1080 x 1920, the middle axis  0.366 -> 0.074 ms
// Bound now: the LDS rows (16 bytes a point) hold ten wavefronts a CU, each one load-to-store chain.
struct R2rMix {
    const double *src;
    double *dst;
    // byte windows around src / dst: the arrays, or (rel) what a workgroup's lines may reach around its first line
    long long src_lo, src_span, dst_lo, dst_span;
    int src_rel, dst_rel;
    LineMap in, out;
    long long sa_in, sa_out;   // element stride along the axis
    long long lines;
    MixShape S;                // M = N/2 points
    const double2 *e1, *e2;    // as R2rParams
    int tb, ld, col, cosine, ortho;
    int in_pairs, out_pairs;   // words 2j, 2j + 1 of every line are one aligned 16-byte word
    double fct;
};

template <int TYPE, class ROW>
__device__ __forceinline__ void r2r_mix_load(const R2rMix &P, long long win, const ROW &row, int base, int i)
{
    const int M = P.S.N, N = 2 * M, NT = P.S.NT;
    const int step = (int)P.sa_in * 8;
    const __amdgpu_buffer_rsrc_t r = make_rsrc((const char *)P.src + win, P.src_span);
    auto pair = [&](int j) -> double2 {   // x[2j], x[2j + 1]
        const int o = base + 2 * j * step;
        return P.in_pairs ? bload2(r, o) : make_double2(bload1(r, o), bload1(r, o + step));
    };
    constexpr int C = 4;   // items in flight per thread
    if constexpr (TYPE == 2) {
        // v[j] = x'[2j], v[N-1-j] = x'[2j+1]; the DST alternates signs
        const double so = P.cosine ? 1.0 : -1.0;
        for (int j0 = i; j0 < M; j0 += C * NT) {
            double2 x[C];
#pragma unroll
            for (int c = 0; c < C; ++c) x[c] = pair(min(j0 + c * NT, M - 1));
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int j = j0 + c * NT;
                if (j < M) {
                    row.word(j) = x[c].x;
                    row.word(N - 1 - j) = so * x[c].y;
                }
            }
        }
    } else if constexpr (TYPE == 3) {
        // z[k] = (V(k) + conj V(M-k)) + i e1[k] (V(k) - conj V(M-k)), V(k) = e2[k] (x'[k] - i x'[N-k]);
        // z[M-k] has the same sum and product conjugated
        const __amdgpu_buffer_rsrc_t r1 = make_rsrc(P.e1, (M + 1LL) * 16), r2 = make_rsrc(P.e2, (M + 1LL) * 16);
        const int o = P.cosine ? 0 : N - 1;   // the ortho end point as the DCT indexes it
        auto off = [&](int n) { return base + (P.cosine ? n : N - 1 - n) * step; };
        const int top = M / 2;
        for (int k0 = i; k0 <= top; k0 += 2 * NT) {
            double x[2][4];
            double2 w1[2], wk[2], wm[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int k = min(k0 + c * NT, top);
                x[c][0] = bload1(r, off(k));
                x[c][1] = bload1(r, off(k ? N - k : N - 1));
                x[c][2] = bload1(r, off(M - k));
                x[c][3] = bload1(r, off(M + k < N ? M + k : N - 1));
                w1[c] = bload2(r1, k * 16);
                wk[c] = bload2(r2, k * 16);
                wm[c] = bload2(r2, (M - k) * 16);
            }
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int k = k0 + c * NT;
                if (k > top) continue;
                double a0 = x[c][0], a1 = k ? x[c][1] : 0.0, b0 = x[c][2], b1 = M + k < N ? x[c][3] : 0.0;
                if (P.ortho) {
                    if (k == o) a0 *= kSqrt2;
                    if (k && N - k == o) a1 *= kSqrt2;
                    if (M - k == o) b0 *= kSqrt2;
                    if (M + k == o) b1 *= kSqrt2;
                }
                const double2 vk = cmul(wk[c], make_double2(a0, -a1));
                const double2 vm = cconj(cmul(wm[c], make_double2(b0, -b1)));
                const double2 s = cadd(vk, vm), d = cmul(w1[c], csub(vk, vm));
                row.at(k) = make_double2(s.x - d.y, s.y + d.x);
                if (k && 2 * k != M) row.at(M - k) = make_double2(s.x + d.y, d.x - s.y);
            }
        }
    } else {
        // z[p] = (x'[2p] + i x'[N-1-2p]) conj(e1[p]) from the words (2p, 2p + 1) and their mirrors
        const __amdgpu_buffer_rsrc_t r1 = make_rsrc(P.e1, (M + 1LL) * 16);
        const int top = (M - 1) / 2;
        for (int p0 = i; p0 <= top; p0 += 2 * NT) {
            double2 a[2], b[2], wa[2], wb[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int p = min(p0 + c * NT, top);
                a[c] = pair(p);
                b[c] = pair(M - 1 - p);
                wa[c] = bload2(r1, p * 16);
                wb[c] = bload2(r1, (M - 1 - p) * 16);
            }
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int p = p0 + c * NT;
                if (p > top) continue;
                // x[2p] = a.x, x[2p+1] = a.y, x[N-2-2p] = b.x, x[N-1-2p] = b.y; the DST reads reversed
                const double2 za = P.cosine ? make_double2(a[c].x, b[c].y) : make_double2(b[c].y, a[c].x);
                const double2 zb = P.cosine ? make_double2(b[c].x, a[c].y) : make_double2(a[c].y, b[c].x);
                row.at(p) = cmul(za, cconj(wa[c]));
                if (2 * p != M - 1) row.at(M - 1 - p) = cmul(zb, cconj(wb[c]));
            }
        }
    }
}

template <int TYPE, class ROW>
__device__ __forceinline__ void r2r_mix_store(const R2rMix &P, long long win, const ROW &row, int base, int i)
{
    const int M = P.S.N, N = 2 * M, NT = P.S.NT;
    const int step = (int)P.sa_out * 8;
    const double f = P.fct;
    const __amdgpu_buffer_rsrc_t r = make_rsrc((char *)P.dst + win, P.dst_span);
    auto put = [&](int n, double v) { bstore1(r, base + n * step, v); };
    auto put_pair = [&](int j, double a, double b) {   // y[2j], y[2j + 1]
        const int o = base + 2 * j * step;
        if (P.out_pairs) {
            bstore2(r, o, make_double2(a, b));
        } else {
            bstore1(r, o, a);
            bstore1(r, o + step, b);
        }
    };
    if constexpr (TYPE == 2) {
        // V[k] = E + conj(e1[k]) O, V[M-k] from the same pair; y[k] = 2 Re, y[N-k] = -2 Im of conj(e2) V
        const __amdgpu_buffer_rsrc_t r1 = make_rsrc(P.e1, (M + 1LL) * 16), r2 = make_rsrc(P.e2, (M + 1LL) * 16);
        const int o = P.cosine ? 0 : N - 1;
        const int top = M / 2;
        auto out = [&](int n, double v) {   // output n as the DCT forms it (the DST stores it reversed)
            if (P.ortho && n == o) v *= 0.5 * kSqrt2;
            put(P.cosine ? n : N - 1 - n, v * f);
        };
        for (int k0 = i; k0 <= top; k0 += 2 * NT) {
            double2 w1[2], wk[2], wm[2], zk[2], zm[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int k = min(k0 + c * NT, top);
                w1[c] = bload2(r1, k * 16);
                wk[c] = bload2(r2, k * 16);
                wm[c] = bload2(r2, (M - k) * 16);
                zk[c] = row.at(k);
                zm[c] = cconj(row.at(k ? M - k : 0));
            }
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int k = k0 + c * NT;
                if (k > top) continue;
                const double2 ev = cscale(cadd(zk[c], zm[c]), 0.5), d = csub(zk[c], zm[c]);
                const double2 od = cmul(cconj(w1[c]), make_double2(0.5 * d.y, -0.5 * d.x));
                const double2 wa = cmul(cconj(wk[c]), cadd(ev, od));
                const double2 wb = cmul(cconj(wm[c]), make_double2(ev.x - od.x, od.y - ev.y));
                out(k, 2.0 * wa.x);
                if (k) out(N - k, -2.0 * wa.y);
                if (2 * k != M) {
                    out(M - k, 2.0 * wb.x);
                    if (k) out(M + k, -2.0 * wb.y);
                }
            }
        }
    } else if constexpr (TYPE == 3) {
        // y[2j] = v[j], y[2j+1] = v[N-1-j], v the real view of the row; the DST alternates signs
        const double so = P.cosine ? f : -f;
        for (int j = i; j < M; j += NT) put_pair(j, f * row.word(j), so * row.word(N - 1 - j));
    } else {
        // S = conj(e2[k]) Z[k]; y[2k] = 2 Re S[k], y[2k+1] = -2 Im S[M-1-k]
        const __amdgpu_buffer_rsrc_t r2 = make_rsrc(P.e2, (M + 1LL) * 16);
        const int top = (M - 1) / 2;
        const double se = 2.0 * f, so = P.cosine ? -2.0 * f : 2.0 * f;
        for (int k0 = i; k0 <= top; k0 += 2 * NT) {
            double2 wa[2], wb[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int k = min(k0 + c * NT, top);
                wa[c] = bload2(r2, k * 16);
                wb[c] = bload2(r2, (M - 1 - k) * 16);
            }
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int k = k0 + c * NT;
                if (k > top) continue;
                const double2 sa = cmul(row.at(k), cconj(wa[c])), sb = cmul(row.at(M - 1 - k), cconj(wb[c]));
                put_pair(k, se * sa.x, so * sb.y);
                if (2 * k != M - 1) put_pair(M - 1 - k, se * sb.x, so * sa.y);
            }
        }
    }
}

template <int TYPE, int WPE, bool PAD>
__global__ void __launch_bounds__(kMixMaxThreads) __attribute__((amdgpu_waves_per_eu(WPE))) k_r2r_mix(const R2rMix P)
{
    using ROW = typename std::conditional<PAD, MixLdsPad, MixLds>::type;
    extern __shared__ double2 zl[];
    __shared__ int off[2][kMaxTB];
    const int tid = (int)threadIdx.x, tb = P.tb, NT = P.S.NT;
    const long long l0 = (long long)xcd_block(blockIdx.x, gridDim.x) * tb;
    const long long wi = P.src_lo + (P.src_rel ? line_off(P.in, l0) * 8 : 0);
    const long long wo = P.dst_lo + (P.dst_rel ? line_off(P.out, l0) * 8 : 0);
    if (tid < tb && l0 + tid < P.lines) {
        off[0][tid] = (int)(line_off(P.in, l0 + tid) * 8 - wi);
        off[1][tid] = (int)(line_off(P.out, l0 + tid) * 8 - wo);
    }
    const int t = P.col ? tid % tb : tid / NT, i = P.col ? tid / tb : tid % NT;
    const bool valid = l0 + t < P.lines;
    const ROW row{zl + t * P.ld};
    __syncthreads();
    if (valid) r2r_mix_load<TYPE>(P, wi, row, off[0][t], i);
    __syncthreads();
    if (P.S.nst) mix_fft<true, true, TYPE == 3 ? 1 : -1>(P.S, row, i, true, row, i, true, 1.0, row, row);
    if (valid) r2r_mix_store<TYPE>(P, wo, row, off[1][t], i);
}

template <int TYPE, int WPE>
static void launch_r2r_mix_tw(const R2rMix &Q, bool pad, unsigned grid, unsigned block, size_t lds, hipStream_t s)
{
    if (pad) hipLaunchKernelGGL((k_r2r_mix<TYPE, WPE, true>), dim3(grid), dim3(block), lds, s, Q);
    else hipLaunchKernelGGL((k_r2r_mix<TYPE, WPE, false>), dim3(grid), dim3(block), lds, s, Q);
}

template <int TYPE>
static hipError_t launch_r2r_mix(const R2rMix &Q, bool pad, unsigned grid, unsigned block, size_t lds, hipStream_t s)
{
    static std::once_flag attr_once;
    std::call_once(attr_once, [] {
        for (const void *f : {(const void *)k_r2r_mix<TYPE, 3, false>, (const void *)k_r2r_mix<TYPE, 3, true>,
                              (const void *)k_r2r_mix<TYPE, 4, false>, (const void *)k_r2r_mix<TYPE, 4, true>})
            if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - 2048) != hipSuccess)
                (void)hipGetLastError();
    });
    if (mix_wpe(grid, block) == 3) launch_r2r_mix_tw<TYPE, 3>(Q, pad, grid, block, lds, s);
    else launch_r2r_mix_tw<TYPE, 4>(Q, pad, grid, block, lds, s);
    return hipGetLastError();
}

static bool smooth13_r2r(long long n)
{
    for (int p : {2, 3, 5, 7, 11, 13})
        while (n % p == 0) n /= p;
    return n == 1;
}

constexpr int kR2rMixMax = 4096;   // longest N/2 of the one-kernel path

// byte window of an array around the pointer, or (rel) around the first line of a workgroup
struct R2rWindow {
    long long lo, span;
    int rel;
};

struct R2r {
    int cosine = 1, type = 2, ortho = 0;
    struct Axis {
        int axis;
        long long N, L, lines;
        int forward, half, col;
        int fused;                        // one kernel (no sub-plan)
        MixShape S;                       // ... its stages, lines per workgroup and LDS row length
        int tb, ld, pad;
        R2rWindow win, wout;              // ... and the arrays around its launches
        std::vector<int> rad;
        std::shared_ptr<DevBuf> tab;      // half lines: e1 | e2 (L + 1 each) | stage twiddles (fused)
        LineMap in_first, in_next, out;
        long long sa_in_first, sa_in_next, sa_out;
        std::unique_ptr<Plan> fft;
    };
    std::vector<Axis> ax;
    DevBuf work;
};

void r2r_destroy(R2r *r) { delete r; }

static LineMap line_map(const std::vector<size_t> &shape, const std::vector<ptrdiff_t> &st, size_t axis)
{
    LineMap m{};
    for (size_t d = 0; d < shape.size(); ++d) {
        if (d == axis) continue;
        m.cnt[m.nd] = (long long)shape[d];
        m.st[m.nd] = (long long)(st[d] / (ptrdiff_t)sizeof(double));
        ++m.nd;
    }
    return m;
}

// the twiddle tables of a half-length axis, from the long-double host generator
static int half_tables(R2r::Axis &A, int type, Error &err)
{
    const long long N = A.N, L = A.L;
    std::vector<double2> t((size_t)(2 * (L + 1))), stages;
    auto cj = [](double2 w) { return make_double2(w.x, -w.y); };   // exp(+i..) from W = exp(-i..)
    for (long long k = 0; k <= L; ++k) {
        if (type == 4) {
            t[(size_t)k] = cj(twiddle_at((uint64_t)k, (uint64_t)(2 * N)));
            t[(size_t)(L + 1 + k)] = cj(twiddle_at((uint64_t)(4 * k + 1), (uint64_t)(8 * N)));
        } else {
            t[(size_t)k] = cj(twiddle_at((uint64_t)k, (uint64_t)N));
            t[(size_t)(L + 1 + k)] = cj(twiddle_at((uint64_t)k, (uint64_t)(4 * N)));
        }
    }
    if (A.fused && !A.rad.empty()) {
        mix_table(stages, A.rad, type == 3 ? 1 : -1);
        t.insert(t.end(), stages.begin(), stages.end());
    }
    A.tab = std::make_shared<DevBuf>();
    if (A.tab->alloc(t.size() * sizeof(double2))) { err = {E_NOMEM, "DCT/DST table allocation failed"}; return E_NOMEM; }
    if (hipMemcpy(A.tab->p, t.data(), t.size() * sizeof(double2), hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipGetLastError();
        err = {E_HIP, "hipMemcpy of a DCT/DST table failed"};
        return E_HIP;
    }
    A.S.tw = (const double2 *)A.tab->p + 2 * (L + 1);
    return OK;
}

// The window of an array [lo, hi) for workgroups of tb lines, whose offsets in it have to fit 31 bits: the
// array itself, or what one workgroup reaches (arrays over 2 GiB).  false: neither fits, and the axis takes
// three passes through a workspace as large as the array.  One kernel against those on one MI355X, DCT-II:
// 33,000 rows of 8,192 (2.2 GB) 1.33 and 3.80 ms, 300,000 of 1,024 1.16 and 4.08, the middle axis of
// 5 x 1,024 x 60,000 1.86 and 4.16.
static bool r2r_window(R2rWindow &w, long long lo, long long hi, const LineMap &m, long long sa, long long N, long long tb)
{
    w = R2rWindow{lo, hi - lo, 0};
    if (w.span <= 0x7fffffff) return true;
    long long a, b;
    line_reach(m, tb, a, b);
    const long long end = (N - 1) * sa;
    a += std::min(end, 0LL);
    b += std::max(end, 0LL);
    w = R2rWindow{a * 8, (b - a + 1) * 8, 1};
    return w.span <= 0x7fffffff;
}

// Threads of a line, where that is more than its butterflies take (16 points a thread): few lines are bound by
// one thread's chain of loads, LDS accesses and butterflies, and many short ones by its unshared
// loads.  Half the points each while the lines then take at most 131,072 threads, else two to eight
// threads along rows and two across them.  MI355X, DCT-II rows: 2,000 x 90 11.4 -> 6.3 us, 100 x 6,250
// 16.3 -> 12.2, 200,000 x 30 68 -> 25 (eight threads 35), 200,000 x 16 27 -> 19; columns 128 x 2,000
// 19 -> 8.0, 30 x 200,000 24.4 -> 23.3 (four threads 25.2).
static long long line_threads(const R2r::Axis &A)
{
    long long half = 1, share = 1;
    while (2 * half < A.L) half *= 2;
    while (2 * share * A.lines <= 131072) share *= 2;
    const long long least = A.col ? (A.L < 10 ? 1 : 2) : A.L < 5 ? 1 : A.L < 8 ? 2 : A.L < 40 ? 4 : 8;
    return std::max(least, std::min(half, share));
}

// The stages, lines per workgroup and LDS rows of the one-kernel path (M = N/2 points): as the
// engine's mixed-radix passes, one line where it fills a wavefront along rows.
static bool mix_axis(const Plan &P, R2r::Axis &A, bool first)
{
    if (!A.half || A.L > kR2rMixMax || !smooth13_r2r(A.L)) return false;
    int nt = 1;
    A.S = MixShape{(int)A.L, 0, 0, 1, nullptr};
    if (A.L > 1) {
        if (!mix_factor((int)A.L, kMixMaxThreads, A.rad, nt, nullptr, 1)) return false;
        if (!A.col && (A.L & (A.L - 1)) == 0) {
            // powers of two along rows: radix-8 stages with one butterfly a thread, twice the wavefronts
            // per LDS row of the radix-16 plan (4096 rows of 4096 points: 86 us with 8 16 16, 68 us so)
            A.rad.clear();
            long long m = A.L;
            while (m % 8 == 0) { A.rad.push_back(8); m /= 8; }
            if (m > 1) A.rad.insert(A.rad.begin(), (int)m);
            nt = (int)std::max<long long>(1, A.L / 8);
        }
        nt = std::max(nt, (int)std::min<long long>(line_threads(A), kMixMaxThreads));
        A.S.NT = nt;
        A.S.nst = (int)A.rad.size();
        for (size_t k = 0; k < A.rad.size(); ++k) A.S.codes |= (unsigned)(A.rad[k] - 1) << (4 * k);
    }
    A.pad = !A.rad.empty() && A.rad[0] % 2 == 0;
    const long long len = A.pad ? A.L + A.L / 16 + 1 : A.L;
    const long long row = len * 16, fit = kMixMaxThreads / nt;
    long long tb;
    if (A.col) {
        // about 40 KiB of LDS a workgroup, four to a CU, and two lines at least: small workgroups
        // overlap one's loads with another's stages (1080-line columns 66 us with four lines of 32-byte
        // runs, 56 us with two; 540-point columns 92 us with eight, 73 us with four).  Lines too long
        // for two take four in one workgroup a CU (2048 points: 248 us alone, 136 with two, 116 with four).
        tb = std::min<long long>(8, 40 * 1024 / row);
        if (tb < 2) tb = 2 * row <= 53 * 1024 ? 2 : std::min<long long>(4, 150 * 1024 / row);
        tb = std::max<long long>(tb, std::min<long long>(256 / nt, 40 * 1024 / row));
    } else {
        tb = nt >= 64 ? 1 : std::min<long long>(128 / nt, 80 * 1024 / row);
    }
    tb = std::min<long long>(std::min<long long>(tb, kMaxTB), fit);
    // small grids are spread over the chip, by whole wavefronts
    const long long wave = std::min<long long>((63 + nt) / nt, tb);
    tb = std::min(tb, std::max({wave, A.col ? 2LL : 1LL, A.lines / 512}));
    tb = std::max<long long>(1, std::min(tb, A.lines));
    if (A.col)
        while (tb & (tb - 1)) tb &= tb - 1;
    const long long in_lo = first ? P.in_lo : P.out_lo, in_hi = first ? P.in_hi : P.out_hi;
    const LineMap &im = first ? A.in_first : A.in_next;
    const long long sa_in = first ? A.sa_in_first : A.sa_in_next;
    while (!r2r_window(A.win, in_lo, in_hi, im, sa_in, A.N, tb) ||
           !r2r_window(A.wout, P.out_lo, P.out_hi, A.out, A.sa_out, A.N, tb)) {
        if (tb == 1) return false;
        tb /= 2;
    }
    if ((A.lines + tb - 1) / tb > 0x7fffffff) return false;
    A.tb = (int)tb;
    A.ld = (int)len;
    if (A.col && tb > 1) {   // lanes across lines meet distinct bank groups
        const int o = tb >= 8 ? 1 : 8 / (int)tb;
        while (A.ld % 8 != o) ++A.ld;
    }
    return true;
}

int r2r_plan_create(std::unique_ptr<Plan> &out, int kind, int type, int ortho, int dtype, size_t ndim,
                    const size_t *shape, const ptrdiff_t *stride_in, const ptrdiff_t *stride_out, size_t naxes,
                    const size_t *axes, Error &err)
{
    if (kind != 5 && kind != 6) { err = {E_INVALID, "unknown transform kind"}; return E_INVALID; }
    if (type < 1 || type > 4) { err = {E_INVALID, kind == 5 ? "invalid DCT type" : "invalid DST type"}; return E_INVALID; }
    if (dtype != 0) { err = {E_UNSUPPORTED, "only IMPULSE_FFT_F64 is supported"}; return E_UNSUPPORTED; }
    if (ndim < 1 || !shape) { err = {E_INVALID, "ndim must be >= 1"}; return E_INVALID; }
    if (ndim > (size_t)kMaxDims) { err = {E_UNSUPPORTED, "too many dimensions"}; return E_UNSUPPORTED; }
    if (!stride_in || !stride_out) { err = {E_INVALID, "stride dimension mismatch"}; return E_INVALID; }
    if (naxes < 1 || !axes) { err = {E_INVALID, "no axes given"}; return E_INVALID; }
    std::vector<int> seen(ndim, 0);
    for (size_t a = 0; a < naxes; ++a) {
        if (axes[a] >= ndim) { err = {E_INVALID, "bad axis number"}; return E_INVALID; }
        if (++seen[axes[a]] > 1) { err = {E_INVALID, "axis specified repeatedly"}; return E_INVALID; }
    }
    int rc = device_check(err);
    if (rc != OK) return rc;
    auto p = std::make_unique<Plan>();
    Plan &P = *p;
    P.kind = kind;
    P.dtype = dtype;
    P.forward = 1;
    (void)hipGetDevice(&P.device);
    P.shape.assign(shape, shape + ndim);
    P.sin.assign(stride_in, stride_in + ndim);
    P.sout.assign(stride_out, stride_out + ndim);
    P.axes.assign(axes, axes + naxes);
    for (size_t d = 0; d < ndim; ++d)
        if (shape[d] == 0) P.empty = true;
    if (P.empty) {
        out = std::move(p);
        return OK;
    }
    for (size_t d = 0; d < ndim; ++d)
        if (P.sin[d] % 8 || P.sout[d] % 8) {
            err = {E_UNSUPPORTED, "strides must be multiples of the element size"};
            return E_UNSUPPORTED;
        }
    plan_spans(P, 8, 8);
    auto R = std::make_unique<R2r>();
    R->cosine = kind == 5;
    R->type = type;
    R->ortho = ortho ? 1 : 0;
    size_t work = 0;
    for (size_t a = 0; a < naxes; ++a) {
        R2r::Axis A;
        A.axis = (int)axes[a];
        A.N = (long long)shape[A.axis];
        if (R->cosine && type == 1 && A.N < 2) {
            err = {E_INVALID, "DCT-I needs at least 2 points along every axis"};
            return E_INVALID;
        }
        A.half = type != 1 && A.N % 2 == 0;
        A.L = A.half ? A.N / 2
                     : (R->cosine && type == 1) ? 2 * (A.N - 1) : (!R->cosine && type == 1) ? 2 * (A.N + 1) : 2 * A.N;
        A.lines = 1;
        for (size_t d = 0; d < ndim; ++d)
            if ((int)d != A.axis) A.lines *= (long long)shape[d];
        A.forward = type != 3;
        A.in_first = line_map(P.shape, P.sin, A.axis);
        A.in_next = line_map(P.shape, P.sout, A.axis);
        A.out = A.in_next;
        A.sa_in_first = P.sin[A.axis] / 8;
        A.sa_in_next = A.sa_out = P.sout[A.axis] / 8;
        // threads walk along lines when the axis is the input's unit-stride dimension, else across lines
        A.col = A.lines > 1 && std::llabs(a == 0 ? A.sa_in_first : A.sa_in_next) != 1;
        A.fused = mix_axis(P, A, a == 0);
        if (A.half && (rc = half_tables(A, type, err)) != OK) return rc;
        if (A.fused) {
            R->ax.push_back(std::move(A));
            continue;
        }
        // c2c over the workspace, in place: [lines, L] along axis 1, or [L, lines] along axis 0
        const size_t fshape_r[2] = {(size_t)A.lines, (size_t)A.L}, fshape_c[2] = {(size_t)A.L, (size_t)A.lines};
        const ptrdiff_t fstr_r[2] = {(ptrdiff_t)(A.L * 16), 16}, fstr_c[2] = {(ptrdiff_t)(A.lines * 16), 16};
        const size_t fax_r[1] = {1}, fax_c[1] = {0};
        rc = A.col ? plan_create(A.fft, 0, 0, 2, fshape_c, fstr_c, fstr_c, 1, fax_c, A.forward, err)
                   : plan_create(A.fft, 0, 0, 2, fshape_r, fstr_r, fstr_r, 1, fax_r, A.forward, err);
        if (rc != OK) return rc;
        work = std::max(work, (size_t)(A.lines * A.L) * sizeof(double2));
        R->ax.push_back(std::move(A));
    }
    if (work && R->work.alloc(work)) { err = {E_NOMEM, "DCT/DST workspace allocation failed"}; return E_NOMEM; }
    P.r2r = R.release();
    out = std::move(p);
    return OK;
}

int r2r_num_launches(const R2r &R)
{
    int n = 0;
    for (const auto &A : R.ax) n += A.fused ? 1 : 2 + (int)A.fft->passes.size();
    return n;
}

// every line starts at an even element
static bool even_lines(const LineMap &m)
{
    for (int d = 0; d < m.nd; ++d)
        if (m.cnt[d] > 1 && m.st[d] % 2) return false;
    return true;
}

int r2r_execute(Plan &P, const void *in, void *out, double fct, hipStream_t s, Error &err)
{
    R2r &R = *P.r2r;
    for (size_t a = 0; a < R.ax.size(); ++a) {
        const auto &A = R.ax[a];
        R2rParams Q;
        Q.src = a == 0 ? (const double *)in : (const double *)out;
        Q.dst = (double *)out;
        Q.work = (double2 *)R.work.p;
        Q.in = a == 0 ? A.in_first : A.in_next;
        Q.out = A.out;
        Q.sa_in = a == 0 ? A.sa_in_first : A.sa_in_next;
        Q.sa_out = A.sa_out;
        Q.N = A.N;
        Q.L = A.L;
        Q.lines = A.lines;
        Q.cosine = R.cosine;
        Q.type = R.type;
        Q.ortho = R.ortho;
        Q.half = A.half;
        Q.col = A.col;
        Q.fct = a == 0 ? fct : 1.0;
        const double2 *tb = A.tab ? (const double2 *)A.tab->p : nullptr;
        Q.e1 = tb;
        Q.e2 = tb ? tb + (A.L + 1) : nullptr;
        if (A.fused) {
            R2rMix F{};
            F.src = Q.src;
            F.dst = Q.dst;
            F.src_lo = A.win.lo;
            F.src_span = A.win.span;
            F.src_rel = A.win.rel;
            F.dst_lo = A.wout.lo;
            F.dst_span = A.wout.span;
            F.dst_rel = A.wout.rel;
            F.in = Q.in;
            F.out = Q.out;
            F.sa_in = Q.sa_in;
            F.sa_out = Q.sa_out;
            F.lines = A.lines;
            F.S = A.S;
            F.e1 = Q.e1;
            F.e2 = Q.e2;
            F.tb = A.tb;
            F.ld = A.ld;
            F.col = A.col && A.tb > 1;
            F.cosine = R.cosine;
            F.ortho = R.ortho;
            F.in_pairs = F.sa_in == 1 && even_lines(F.in) && (uintptr_t)F.src % 16 == 0;
            F.out_pairs = F.sa_out == 1 && even_lines(F.out) && (uintptr_t)F.dst % 16 == 0;
            F.fct = Q.fct;
            const unsigned grid = (unsigned)((A.lines + A.tb - 1) / A.tb), block = (unsigned)(A.tb * A.S.NT);
            const size_t lds = (size_t)A.ld * (size_t)A.tb * sizeof(double2);
            hipError_t e = R.type == 2   ? launch_r2r_mix<2>(F, A.pad, grid, block, lds, s)
                           : R.type == 3 ? launch_r2r_mix<3>(F, A.pad, grid, block, lds, s)
                                         : launch_r2r_mix<4>(F, A.pad, grid, block, lds, s);
            if (e != hipSuccess) { err = {E_HIP, std::string("DCT/DST launch: ") + hipGetErrorString(e)}; return E_HIP; }
            continue;
        }
        const long long pre = A.lines * A.L, post = A.lines * r2r_post_count(A.half, R.type, A.N);
        const unsigned gpre = (unsigned)std::min<long long>((pre + 255) / 256, 1 << 20);
        const unsigned gpost = (unsigned)std::min<long long>((post + 255) / 256, 1 << 20);
        hipLaunchKernelGGL(k_r2r_pre, dim3(gpre), dim3(256), 0, s, Q);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) { err = {E_HIP, std::string("DCT/DST launch: ") + hipGetErrorString(e)}; return E_HIP; }
        int rc = plan_execute(*A.fft, R.work.p, R.work.p, 1.0, s, err);
        if (rc != OK) return rc;
        hipLaunchKernelGGL(k_r2r_post, dim3(gpost), dim3(256), 0, s, Q);
        e = hipGetLastError();
        if (e != hipSuccess) { err = {E_HIP, std::string("DCT/DST launch: ") + hipGetErrorString(e)}; return E_HIP; }
    }
    return OK;
}

}  // namespace ifft
