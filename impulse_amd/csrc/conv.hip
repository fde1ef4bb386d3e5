// FFT-based 2-D convolution with a reverse-mode backward pass.
//
// Forward ("same" output, kernel origin at its centre c = ((KH-1)/2, (KW-1)/2)):
//   y_b = crop_c( c2r( K^ . r2c(pad_0 x_b) ) ) / (P Q),   K^ = r2c(pad_0 k)
// on a P x Q grid, P >= H + KH - 1 and Q >= W + KW - 1 (13-smooth, Q even).
// Backward, written with the adjoint of every step (pad* = crop, crop* = pad,
// (K^ .)* = conj(K^) ., r2c* / c2r* = the R2C_ADJOINT / C2R_ADJOINT plans):
//   G_b  = c2r*( pad_c g_b ) / (P Q)
//   gx_b = crop_0( r2c*( conj(K^) . G_b ) )
//   gk   = crop_0( r2c*( sum_b conj(X^_b) . G_b ) )
// The spectra X^_b and K^ are recomputed in the backward pass instead of being
// stored by the forward pass.  Inputs and outputs are float32 or float64; all
// arithmetic is FP64.
//
// Fused path (grids with P <= 2560 and Q/2 <= 2560): three kinds of mixed-radix kernels (mix_fft.h)
// over half spectra, and only for the rows an image occupies:
//   rows   : real rows read straight from the caller's array (the padding is
//            generated, never stored), r2c of length Q by the half-length
//            complex transform, half spectrum out;
//   columns: each workgroup loads its columns' image rows at their grid offset (the
//            other P - H rows are zeros), transforms, multiplies by K^ (conj K^ for
//            the adjoint) and transforms back in one kernel, keeping only the
//            rows the crop needs -- or, for the kernel gradient, sums
//            conj(X^_b) G^_b over the images of a chunk;
//   rows^-1: c2r of the kept rows, the cropped columns scaled and stored in the
//            caller's dtype.
// Three passes over half spectra instead of pad / r2c / multiply / c2r / crop
// over the whole padded grid.  Larger grids take the plan-based path.
//
// The half spectra are kept in column blocks, S[img][block][row][cb] with cb neighbouring columns
// (the columns of one workgroup): a column workgroup reads and writes one contiguous run of
// memory, and a row workgroup of several rows writes rows cb 16 bytes at a time.
//
// Measured on one MI355X, 16 x 2048^2 images and a 63 x 63 kernel in float32 (grid 2160 x 2100),
// against LDS kernels that staged every point at both ends: rows 0.41 -> 0.25 ms (0.82 GB moved),
// columns of the convolution 1.04 -> 0.31 ms (1.10 GB), of the kernel gradient 1.21 -> 0.57 ms (1.10
// GB), rows^-1 0.35 -> 0.26 ms; forward and backward together 5.2 -> 2.6 ms.  Bounds now: the
// convolution's columns move their bytes at 3.5 TB/s with VALU issue at 40 %; the rows are held by
// LDS (67 KB, two workgroups a CU); the kernel gradient's image loop serialises its loads with its
// barriers, at 12 wavefronts a CU.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <initializer_list>
#include <vector>

#include "engine.h"
#include "fft_common.h"
#include "mix_fft.h"

namespace ifft {

// dst[b, i, j] (P x Q, f64) = src[b, i - oy, j - ox] for the in-range part, else 0
template <typename T>
__global__ void k_pad2d(const T *__restrict__ src, double *__restrict__ dst, int B, int H, int W, int P, int Q, int oy,
                        int ox)
{
    const long long total = (long long)B * P * Q;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (long long)gridDim.x * blockDim.x) {
        const int j = (int)(e % Q);
        const long long r = e / Q;
        const int i = (int)(r % P);
        const int b = (int)(r / P);
        const int si = i - oy, sj = j - ox;
        double v = 0.0;
        if (si >= 0 && si < H && sj >= 0 && sj < W) v = (double)src[((long long)b * H + si) * W + sj];
        dst[e] = v;
    }
}

// dst[b, i, j] = scale * src[b, i + oy, j + ox], i < H, j < W
template <typename T>
__global__ void k_crop2d(const double *__restrict__ src, T *__restrict__ dst, int B, int H, int W, int P, int Q, int oy,
                         int ox, double scale)
{
    const long long total = (long long)B * H * W;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (long long)gridDim.x * blockDim.x) {
        const int j = (int)(e % W);
        const long long r = e / W;
        const int i = (int)(r % H);
        const int b = (int)(r / H);
        dst[e] = (T)(scale * src[((long long)b * P + i + oy) * Q + j + ox]);
    }
}

// z[b, m] = a[b, m] * (conj ? conj(k[m]) : k[m]), m < n
__global__ void k_spec_mul(const double2 *__restrict__ a, const double2 *__restrict__ k, double2 *__restrict__ z, int B,
                           long long n, int conj)
{
    const long long total = (long long)B * n;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (long long)gridDim.x * blockDim.x) {
        const double2 kv = k[e % n];
        z[e] = cmul(a[e], conj ? cconj(kv) : kv);
    }
}

// r[m] = sum_b conj(a[b, m]) * g[b, m]
__global__ void k_spec_corr_reduce(const double2 *__restrict__ a, const double2 *__restrict__ g, double2 *__restrict__ r,
                                   int B, long long n)
{
    for (long long m = (long long)blockIdx.x * blockDim.x + threadIdx.x; m < n; m += (long long)gridDim.x * blockDim.x) {
        double2 acc = make_double2(0.0, 0.0);
        for (int b = 0; b < B; ++b) acc = cadd(acc, cmul(cconj(a[(long long)b * n + m]), g[(long long)b * n + m]));
        r[m] = acc;
    }
}

// ---------------------------------------------------------------------------
// fused path
// ---------------------------------------------------------------------------

constexpr int kConvThreads = 512;      // workgroup size cap of the fused kernels
constexpr int kConvMaxLen = 2560;      // longest rows (complex points) and columns of the fused path
constexpr int kConvMaxTb = 64;         // rows per workgroup of the row kernels at most
constexpr int kConvAcc = 8;            // kernel-gradient sums a thread holds (P / 2 points over NT threads)

// half spectra in column blocks: element (img, row, j) of `rows` rows per image
struct ConvSpec {
    double2 *p;
    int rows, nblk, lcb;   // rows per image, blocks per row, log2 of the columns per block
    __device__ __forceinline__ long long block(long long img, int blk) const
    {
        return ((img * nblk + blk) * rows) << lcb;
    }
};

// real rows -> half spectra: row q of src (W values, placed at grid columns
// [rx, rx + W) of a 2 M-point row, zeros elsewhere) -> S(q, 0 .. M)
struct ConvRowSet {
    const void *src;
    ConvSpec S;
    long long rows;       // rows of all images
    long long span;       // bytes a workgroup's rows may reach from their first image on
    int W, rx;
    unsigned groups;      // workgroups of this set
};
// Up to three sets of rows share one launch: the few rows of the convolution kernel would take a
// launch of their own 44 us (one workgroup's latency) beside the 250 us of the images' rows.
struct ConvRows {
    ConvRowSet set[3];
    MixShape F;
    const double2 *rtw;   // W_{2M}^k, k <= M / 2
    int nset, f32, ltb;   // ltb: log2 of the rows per workgroup
};

// half spectra -> real rows: S(q, 0 .. M) -> dst[q][c] = scale * x[ox + c], c < Wout,
// x the unnormalised c2r of length 2 M
struct ConvRowInvSet {
    ConvSpec S;
    void *dst;
    long long rows, span;
    int Wout, ox;
    unsigned groups;
};
struct ConvRowsInv {
    ConvRowInvSet set[2];
    MixShape F;
    const double2 *rtw;
    int nset, f32, ltb;
    double scale;
};

// column passes over blocks of cb columns (grid rows 0 .. P-1, image rows at [r0, r0 + S.rows))
struct ConvCols {
    ConvSpec Sa, Sg;       // image rows; gradient rows (kernel gradient)
    ConvSpec So;           // kept rows: grid rows [oy, oy + So.rows)
    double2 *KT;           // kernel spectrum [block][P][cb]
    double2 *acc;          // kernel-gradient partial sums [chunk][block][P][cb]
    MixShape F, I;         // forward, and the inverse with reversed radices
    int ra, rg, oy, nimg, chunk, nchunk, conjk, sub;
};

enum ConvColMode { CC_SPECTRUM = 0, CC_CONV = 1, CC_GK = 2, CC_GK_FINAL = 3 };

// 32-bit offset that a buffer access never finds in range: loads give zero, stores are dropped
constexpr int kNowhere = 0x7ffffff0;

struct ConvRowIn {
    __amdgpu_buffer_rsrc_t r;
    int base, W, rx, f32;   // element offset of the row in the window (kNowhere / 16: no row)
    bool pairs;             // both words of a point sit in one aligned complex word, or are both outside
    template <int R> __device__ __forceinline__ void load(double2 *v, int b, int nb) const
    {
        if (pairs && f32) {
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const int c = 2 * (b + q * nb) - rx;
                const float2 f = bloadf2(r, (unsigned)c < (unsigned)W ? (base + c) * 4 : kNowhere);
                v[q] = make_double2((double)f.x, (double)f.y);
            }
        } else if (pairs) {
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const int c = 2 * (b + q * nb) - rx;
                v[q] = bload2(r, (unsigned)c < (unsigned)W ? (base + c) * 8 : kNowhere);
            }
        } else if (f32) {
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const int c = 2 * (b + q * nb) - rx;
                v[q] = make_double2((double)bloadf1(r, (unsigned)c < (unsigned)W ? (base + c) * 4 : kNowhere),
                                    (double)bloadf1(r, (unsigned)(c + 1) < (unsigned)W ? (base + c + 1) * 4 : kNowhere));
            }
        } else {
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const int c = 2 * (b + q * nb) - rx;
                v[q] = make_double2(bload1(r, (unsigned)c < (unsigned)W ? (base + c) * 8 : kNowhere),
                                    bload1(r, (unsigned)(c + 1) < (unsigned)W ? (base + c + 1) * 8 : kNowhere));
            }
        }
    }
};

// byte offset of row `row`'s first bin from the start of image img0
__device__ __forceinline__ int conv_row_off(const ConvSpec &S, long long row, long long img0)
{
    const long long img = row / S.rows;
    const int r = (int)(row - img * S.rows);
    return (int)((S.block(img, 0) - S.block(img0, 0) + ((long long)r << S.lcb)) * 16);
}
// byte offset of bin k from its row's first bin
__device__ __forceinline__ int conv_bin_off(const ConvSpec &S, int k)
{
    return (((k >> S.lcb) * S.rows << S.lcb) + (k & ((1 << S.lcb) - 1))) * 16;
}

template <int WPE>
__global__ void __launch_bounds__(kConvThreads) __attribute__((amdgpu_waves_per_eu(WPE))) k_conv_rows(const ConvRows P)
{
    extern __shared__ double2 zl[];
    __shared__ int roff[kConvMaxTb];
    const int tid = (int)threadIdx.x, M = P.F.N, NT = P.F.NT, tb = 1 << P.ltb;
    unsigned blk = xcd_block(blockIdx.x, gridDim.x);
    int which = 0;
    while (which + 1 < P.nset && blk >= P.set[which].groups) blk -= P.set[which++].groups;
    const ConvRowSet &A = P.set[which];
    const ConvSpec S = A.S;
    const long long q0 = (long long)blk * tb;
    const int t = tid / NT, i = tid - t * NT;
    const int es = P.f32 ? 4 : 8;
    const int nrow = (int)(A.rows - q0 < tb ? A.rows - q0 : tb);
    const long long img0 = q0 / S.rows;
    if (tid < nrow) roff[tid] = conv_row_off(S, q0 + tid, img0);
    ConvRowIn in;
    in.r = make_rsrc((const char *)A.src + q0 * A.W * es, (long long)nrow * A.W * es);
    in.base = t * A.W;
    in.W = t < nrow ? A.W : 0;
    in.rx = A.rx;
    in.f32 = P.f32;
    in.pairs = !(A.rx & 1) && !(A.W & 1) && (uintptr_t)A.src % (2 * es) == 0;
    double2 *row = zl + t * M;
    mix_fft<false, true, -1>(P.F, MixLds{row}, i, true, MixLds{row}, i, true, -1.0, in, MixLds{row});   // ends with a barrier
    // X[k] = E + W_{2M}^k O and X[M-k] = conj(E) - conj(W^k O), E = (Z[k] + conj Z[M-k]) / 2,
    // O = (Z[k] - conj Z[M-k]) / 2i.  Lanes walk a block's columns, then the rows; four bin pairs
    // in flight per thread.
    const int nthr = tb * NT, lc = S.lcb + P.ltb;
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(P.rtw, ((long long)(M / 2) + 1) * 16);
    const __amdgpu_buffer_rsrc_t ro = make_rsrc(S.p + S.block(img0, 0), A.span);
    const int top = M / 2;
    const int total = ((top >> S.lcb) + 1) << lc;   // whole blocks of bins
    for (int e0 = tid; e0 < total; e0 += 4 * nthr) {
        double2 w[4], z[4], m[4];
        int kk[4], tt[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int e = e0 + c * nthr;
            tt[c] = (e >> S.lcb) & (tb - 1);
            kk[c] = (e >> lc << S.lcb) + (e & ((1 << S.lcb) - 1));
            const int k = min(kk[c], top);
            w[c] = bload2(rw, k * 16);
            const double2 *zr = zl + tt[c] * M;
            z[c] = zr[k];
            m[c] = zr[k ? M - k : 0];
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int k = kk[c], km = M - k;
            if (k > top || tt[c] >= nrow) continue;
            const double2 zm = cconj(m[c]);
            const double2 ev = cscale(cadd(z[c], zm), 0.5), d = csub(z[c], zm);
            const double2 o = cmul(make_double2(0.5 * d.y, -0.5 * d.x), w[c]);
            const int off = roff[tt[c]];
            bstore2(ro, off + conv_bin_off(S, k), cadd(ev, o));
            bstore2(ro, off + conv_bin_off(S, km), make_double2(ev.x - o.x, o.y - ev.y));
        }
    }
}

struct ConvRowOut {
    __amdgpu_buffer_rsrc_t r;
    int base, Wout, ox, f32;
    double f;
    template <int R, class G> __device__ __forceinline__ void store(const double2 *v, int n, int dn, G) const
    {
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const int c = 2 * (n + q * dn) - ox;
            const bool a = (unsigned)c < (unsigned)Wout, b = (unsigned)(c + 1) < (unsigned)Wout;
            if (f32) {
                bstoref1(r, a ? (base + c) * 4 : kNowhere, f * v[q].x);
                bstoref1(r, b ? (base + c + 1) * 4 : kNowhere, f * v[q].y);
            } else {
                bstore1(r, a ? (base + c) * 8 : kNowhere, f * v[q].x);
                bstore1(r, b ? (base + c + 1) * 8 : kNowhere, f * v[q].y);
            }
        }
    }
};

template <int WPE>
__global__ void __launch_bounds__(kConvThreads) __attribute__((amdgpu_waves_per_eu(WPE))) k_conv_rows_inv(const ConvRowsInv P)
{
    extern __shared__ double2 zl[];
    __shared__ int roff[kConvMaxTb];
    const int tid = (int)threadIdx.x, M = P.F.N, NT = P.F.NT, tb = 1 << P.ltb;
    unsigned blk = xcd_block(blockIdx.x, gridDim.x);
    int which = 0;
    while (which + 1 < P.nset && blk >= P.set[which].groups) blk -= P.set[which++].groups;
    const ConvRowInvSet &A = P.set[which];
    const ConvSpec S = A.S;
    const long long q0 = (long long)blk * tb;
    const int nrow = (int)(A.rows - q0 < tb ? A.rows - q0 : tb);
    const long long img0 = q0 / S.rows;
    if (tid < nrow) roff[tid] = conv_row_off(S, q0 + tid, img0);
    __syncthreads();
    const int nthr = tb * NT, lc = S.lcb + P.ltb;
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(P.rtw, ((long long)(M / 2) + 1) * 16);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(S.p + S.block(img0, 0), A.span);
    const int top = M / 2;
    const int total = ((top >> S.lcb) + 1) << lc;
    // Z[k] = E + i O, E = X[k] + conj X[M-k], O = (X[k] - conj X[M-k]) conj(W^k), and Z[M-k] =
    // conj(E) + i conj(O); the imaginary parts of X[0] and X[M] are ignored, as c2r does
    for (int e0 = tid; e0 < total; e0 += 4 * nthr) {
        double2 w[4], x[4], m[4];
        int kk[4], tt[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int e = e0 + c * nthr;
            tt[c] = (e >> S.lcb) & (tb - 1);
            kk[c] = (e >> lc << S.lcb) + (e & ((1 << S.lcb) - 1));
            const int k = min(kk[c], top);
            const int off = tt[c] < nrow ? roff[tt[c]] : kNowhere / 2;
            w[c] = bload2(rw, k * 16);
            x[c] = bload2(rs, off + conv_bin_off(S, k));
            m[c] = bload2(rs, off + conv_bin_off(S, M - k));
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int k = kk[c];
            if (k > top || tt[c] >= nrow) continue;
            double2 a = x[c], b = m[c];
            if (k == 0) a.y = b.y = 0.0;
            const double2 ev = cadd(a, cconj(b)), o = cmul(csub(a, cconj(b)), cconj(w[c]));
            double2 *zr = zl + tt[c] * M;
            zr[k] = make_double2(ev.x - o.y, ev.y + o.x);
            if (k && 2 * k != M) zr[M - k] = make_double2(ev.x + o.y, o.x - ev.y);
        }
    }
    __syncthreads();
    const int t = tid / NT, i = tid - t * NT;
    const int es = P.f32 ? 4 : 8;
    double2 *row = zl + t * M;
    ConvRowOut out;
    out.r = make_rsrc((char *)A.dst + q0 * A.Wout * es, (long long)nrow * A.Wout * es);
    out.base = t * A.Wout;
    out.Wout = t < nrow ? A.Wout : 0;
    out.ox = A.ox;
    out.f32 = P.f32;
    out.f = P.scale;
    mix_fft<true, false, 1>(P.F, MixLds{row}, i, true, MixLds{row}, i, true, 1.0, MixLds{row}, out);
}

// column `t` of a block: rows [r0, r0 + rows) of the grid, zeros elsewhere
struct ConvColIn {
    __amdgpu_buffer_rsrc_t r;
    int t, lcb, rows, r0;
    template <int R> __device__ __forceinline__ void load(double2 *v, int b, int nb) const
    {
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const int m = b + q * nb - r0;
            v[q] = bload2(r, (unsigned)m < (unsigned)rows ? ((m << lcb) + t) * 16 : kNowhere);
        }
    }
};

// the same from a pointer of the thread's own (x and g columns side by side in one workgroup)
struct ConvColIn2 {
    const double2 *col;
    int lcb, rows, r0;
    template <int R> __device__ __forceinline__ void load(double2 *v, int b, int nb) const
    {
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const int m = b + q * nb - r0;
            const bool ok = (unsigned)m < (unsigned)rows;
            const double2 x = col[(ok ? m : 0) << lcb];
            v[q] = ok ? x : make_double2(0.0, 0.0);
        }
    }
};

// grid rows [oy, oy + rows) of column `t`
struct ConvColOut {
    __amdgpu_buffer_rsrc_t r;
    int t, lcb, rows, oy;
    template <int R, class G> __device__ __forceinline__ void store(const double2 *v, int n, int dn, G) const
    {
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const int m = n + q * dn - oy;
            bstore2(r, (unsigned)m < (unsigned)rows ? ((m << lcb) + t) * 16 : kNowhere, v[q]);
        }
    }
};

// v[q] times K^ (or conj K^) at column positions b + q nb
struct ConvColMul {
    __amdgpu_buffer_rsrc_t r;
    int t, lcb;
    double cj;
    template <int R> __device__ __forceinline__ void apply(double2 *v, int b, int nb) const
    {
#pragma unroll
        for (int q = 0; q < R; ++q) {
            double2 k = bload2(r, (((b + q * nb) << lcb) + t) * 16);
            k.y *= cj;
            v[q] = cmul(v[q], k);
        }
    }
};

// sum of the chunks' partial spectra of column `t`
struct ConvAccIn {
    const double2 *acc;
    long long step;   // elements from one chunk to the next
    int n, t, lcb;
    template <int R> __device__ __forceinline__ void load(double2 *v, int b, int nb) const
    {
#pragma unroll
        for (int q = 0; q < R; ++q) v[q] = make_double2(0.0, 0.0);
        // a few chunks' loads in flight, added in their order
        constexpr int U = R > 4 ? 1 : R > 2 ? 2 : 4;
        int c = 0;
        for (; c + U <= n; c += U) {
            double2 x[U][R];
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int q = 0; q < R; ++q) x[u][q] = acc[(c + u) * step + ((b + q * nb) << lcb) + t];
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int q = 0; q < R; ++q) v[q] = cadd(v[q], x[u][q]);
        }
        for (; c < n; ++c)
#pragma unroll
            for (int q = 0; q < R; ++q) v[q] = cadd(v[q], acc[c * step + ((b + q * nb) << lcb) + t]);
    }
};

template <int MODE, int WPE>
__global__ void __launch_bounds__(MODE == CC_GK && WPE == 4 ? 2 * kConvThreads : kConvThreads)
__attribute__((amdgpu_waves_per_eu(WPE))) k_conv_cols(const ConvCols C)
{
    extern __shared__ double2 zl[];
    const int P = C.F.N, NT = C.F.NT, lcb = C.Sa.lcb, cb = 1 << lcb, nblk = C.Sa.nblk;
    const int tid = (int)threadIdx.x;
    const unsigned logical = xcd_block(blockIdx.x, gridDim.x);
    // LDS row stride: lanes that walk across columns meet distinct bank groups
    const int cols = MODE == CC_GK ? 2 * C.sub : cb;
    const int t = tid & (cols - 1), i = tid / cols;
    const int ld = cols > 1 ? P + ((8 / cols - P) & 7) : P;
    double2 *row = zl + t * ld;
    const long long span = ((long long)P << lcb) * 16;   // one block of kernel or partial spectrum

    if constexpr (MODE == CC_SPECTRUM) {
        const int blk = (int)logical;
        const ConvColIn in{make_rsrc(C.Sa.p + C.Sa.block(0, blk), ((long long)C.Sa.rows << lcb) * 16), t, lcb, C.Sa.rows, C.ra};
        const ConvColOut out{make_rsrc(C.KT + ((long long)blk * P << lcb), span), t, lcb, P, 0};
        mix_fft<false, false, -1>(C.F, MixLds{row}, i, true, MixLds{row}, i, true, -1.0, in, out);
    } else if constexpr (MODE == CC_CONV) {
        // images fastest: neighbouring workgroups share their block of K^ in the L2
        const int img = (int)(logical % (unsigned)C.nimg), blk = (int)(logical / (unsigned)C.nimg);
        const ConvColIn in{make_rsrc(C.Sa.p + C.Sa.block(img, blk), ((long long)C.Sa.rows << lcb) * 16), t, lcb, C.Sa.rows, C.ra};
        const ConvColMul mul{make_rsrc(C.KT + ((long long)blk * P << lcb), span), t, lcb, C.conjk ? -1.0 : 1.0};
        const ConvColOut out{make_rsrc(C.So.p + C.So.block(img, blk), ((long long)C.So.rows << lcb) * 16), t, lcb, C.So.rows, C.oy};
        mix_conv(C.F, C.I, row, i, in, mul, out);
    } else if constexpr (MODE == CC_GK) {
        // x and g columns transformed together (slots 0 .. sub-1 and sub .. 2 sub - 1), `sub` columns
        // of a block per workgroup; the chunk's sum of conj(X^) G^ in registers
        const int nsub = cb / C.sub;
        const int part = (int)(logical % (unsigned)nsub);
        const int blk = (int)(logical / (unsigned)nsub % (unsigned)nblk), chunk = (int)(logical / (unsigned)(nsub * nblk));
        const bool isg = t >= C.sub;
        const int nthr = cols * NT, n = C.sub * P;
        double2 acc[kConvAcc];
#pragma unroll
        for (int q = 0; q < kConvAcc; ++q) acc[q] = make_double2(0.0, 0.0);
        const int b1 = min(C.nimg, (chunk + 1) * C.chunk);
        for (int b = chunk * C.chunk; b < b1; ++b) {
            const ConvColIn2 in{(isg ? C.Sg.p : C.Sa.p) + C.Sa.block(b, blk) + part * C.sub + (t & (C.sub - 1)), lcb,
                                C.Sa.rows, isg ? C.rg : C.ra};
            mix_fft<false, true, -1>(C.F, MixLds{row}, i, true, MixLds{row}, i, true, -1.0, in, MixLds{row});
            const int e0 = opaque(tid);   // the LDS addresses are not worth registers across the transform
#pragma unroll
            for (int q = 0; q < kConvAcc; ++q) {
                const int e = e0 + q * nthr;
                if (e < n) {
                    const int tt = e & (C.sub - 1), m = e / C.sub;
                    acc[q] = cadd(acc[q], cmul(cconj(zl[tt * ld + m]), zl[(C.sub + tt) * ld + m]));
                }
            }
            __syncthreads();
        }
        double2 *out = C.acc + ((((long long)chunk * nblk + blk) * P) << lcb);
#pragma unroll
        for (int q = 0; q < kConvAcc; ++q) {
            const int e = tid + q * nthr;
            if (e < n) out[((e / C.sub) << lcb) + part * C.sub + (e & (C.sub - 1))] = acc[q];
        }
    } else {   // CC_GK_FINAL
        const int blk = (int)logical;
        const ConvAccIn in{C.acc + ((long long)blk * P << lcb), (long long)nblk * P << lcb, C.nchunk, t, lcb};
        const ConvColOut out{make_rsrc(C.So.p + C.So.block(0, blk), ((long long)C.So.rows << lcb) * 16), t, lcb, C.So.rows, C.oy};
        mix_fft<false, false, 1>(C.F, MixLds{row}, i, true, MixLds{row}, i, true, 1.0, in, out);
    }
}

static MixShape mix_shape(int N, const std::vector<int> &rad, int nt, const double2 *tw)
{
    MixShape S{N, (int)rad.size(), 0, nt, tw};
    for (size_t k = 0; k < rad.size(); ++k) S.codes |= (unsigned)(rad[k] - 1) << (4 * k);
    return S;
}

static unsigned blocks_for(long long total)
{
    long long b = (total + 255) / 256;
    return (unsigned)std::max<long long>(1, std::min<long long>(b, 1 << 16));
}

static bool smooth13_c(long long n)
{
    for (int p : {2, 3, 5, 7, 11, 13})
        while (n % p == 0) n /= p;
    return n == 1;
}

static long long conv_len(long long need, bool even)
{
    for (long long n = need;; ++n)
        if ((!even || n % 2 == 0) && smooth13_c(n) && (!even || smooth13_c(n / 2))) return n;
}

struct Conv2d {
    int B = 0, H = 0, W = 0, KH = 0, KW = 0, dtype = 0;   // dtype 0: f64, 1: f32
    long long P = 0, Q = 0, nspec = 0;                     // grid and half-spectrum points per image
    // plan-based path (grids beyond the fused kernels)
    std::unique_ptr<Plan> r2c_b, r2c_1, c2r_b, c2r_adj_b, r2c_adj_b, r2c_adj_1;
    DevBuf pad, spec_a, spec_b, kspec, kpad;
    // fused path
    bool fused = false;
    int lcb = 0, ltb = 0, sub = 1, nblk = 1, nchunk = 1, chunk = 1;
    MixShape Ff{}, Fi{};    // columns: forward, inverse with reversed radices
    MixShape Rf{}, Ri{};    // rows: forward, inverse
    DevBuf tab;             // their stage tables and W_Q^k, k <= Q/4
    const double2 *rtw = nullptr;
    DevBuf sx, sg, sk, kt;  // half spectra of the images (two) and of the kernel rows, kernel spectrum
    DevBuf acc;             // kernel-gradient partial sums [nchunk][block][P][cb]
};

// the cheapest length of at least `need` points the mixed-radix stages take (within 1/16, or the
// first one found), by the operation count of a whole transform
static long long conv_fused_len(long long need)
{
    long long best = 0;
    double cost = 0.0;
    for (long long n = std::max<long long>(need, 4); n <= kConvMaxLen; ++n) {
        if (best && n > need + need / 16) break;
        std::vector<int> rad;
        int nt;
        double c;
        if (!smooth13_c(n) || !mix_factor((int)n, kConvThreads / 2, rad, nt, &c)) continue;
        if (!best || c < cost) {
            best = n;
            cost = c;
        }
    }
    return best;
}

// Fused path set-up for grids the kernels hold: block widths, image chunks,
// tables and workspaces.  Leaves c.fused false for larger grids.
static int conv_fused_setup(Conv2d &c, Error &err)
{
    // A circular convolution of period P gives the 'same' rows [cy, cy + H) of the linear one when
    // P >= H + max(cy, KH - 1 - cy): the wrapped terms then only touch rows the crop drops.  The
    // correlations of the backward pass need the same bound (their wrapped terms land outside
    // [0, KH) and [0, H)).  Likewise for the columns.
    const int cy = (c.KH - 1) / 2, cx = (c.KW - 1) / 2;
    const long long P = conv_fused_len((long long)c.H + std::max(cy, c.KH - 1 - cy));
    const long long M = conv_fused_len(((long long)c.W + std::max(cx, c.KW - 1 - cx) + 1) / 2), Qh = M + 1;
    if (!P || !M) return OK;
    std::vector<int> rc, rr;
    int ntc = 0, ntr = 0;
    if (!mix_factor((int)P, kConvThreads / 2, rc, ntc) || !mix_factor((int)M, kConvThreads / 2, rr, ntr)) return OK;
    c.P = P;
    c.Q = 2 * M;
    c.nspec = c.P * Qh;
    // Columns per block: a wavefront's worth of threads.  One column where it fills one leaves
    // small workgroups, several to a CU (backward of 8 x 1024^2, 31 x 31: 0.304 ms with four columns,
    // 0.257 ms with one); half-filled wavefronts cost more than that (21 x 439 x 1713, 13 x 9: 448
    // points by 32 threads, forward 0.221 -> 0.255 ms).  The kernel gradient holds x and g columns.
    const long long lds = 80 * 1024 - 1024;
    while (c.lcb < 3 && (1 << c.lcb) * ntc < 64 && (2LL << c.lcb) * (P + 8) * 16 <= lds) ++c.lcb;
    // Short columns: threads beyond 16 points each until the block fills a wavefront, one per butterfly at
    // most (kernel gradient of 2,000 x 16^2 images, 3 x 3: 162 -> 101 us, forward 38.7 -> 33.3).
    int widest = 1;
    for (int r : rc) widest = std::max(widest, (int)(P / r));
    ntc = std::max(ntc, std::min(64 >> c.lcb, widest));
    c.sub = std::max(1, (1 << c.lcb) / 2);
    c.nblk = (int)((Qh + (1 << c.lcb) - 1) >> c.lcb);
    // rows per workgroup: whole 128-byte lines of a block, a wavefront at least
    while ((1 << (c.lcb + c.ltb)) * 16 < 128 || (1 << c.ltb) * ntr < 64) {
        if ((2LL << c.ltb) * M * 16 > lds || (2 << c.ltb) * ntr > kConvThreads || (2 << c.ltb) > kConvMaxTb) break;
        ++c.ltb;
    }
    // Kernel gradient: chunks of images that make three rounds of two workgroups per CU.  A workgroup sums
    // its chunk's images one after the other and the final pass the chunks, so batches of many small
    // images balance the two: 1.75 sqrt(B) chunks at most, and eight for any batch.  Times with 8, 1.75
    // sqrt(B) and 4 sqrt(B) chunks (MI355X, f32): 2,000 x 16^2, 3 x 3 540, 90 and 98 us; 100 x 28^2, 7 x 7
    // 88, 83 and 105; 256 x 64^2, 9 x 9 157, 115 and 140.
    const long long ng = (long long)c.nblk * ((1 << c.lcb) / c.sub);
    const int most = std::max(8, (int)(1.75 * std::sqrt((double)c.B)));
    c.nchunk = (int)std::max<long long>(1, std::min<long long>(std::min(c.B, most), (3 * 512 + ng - 1) / ng));
    c.chunk = (c.B + c.nchunk - 1) / c.nchunk;
    c.nchunk = (c.B + c.chunk - 1) / c.chunk;
    // tables
    std::vector<double2> all, h;
    size_t at[5];
    std::vector<int> rci(rc.rbegin(), rc.rend());
    auto add = [&](size_t k) { at[k] = all.size(); all.insert(all.end(), h.begin(), h.end()); };
    mix_table(h, rc, -1); add(0);
    mix_table(h, rci, 1); add(1);
    mix_table(h, rr, -1); add(2);
    mix_table(h, rr, 1); add(3);
    twiddle_table(h, (uint64_t)c.Q, (uint64_t)(M / 2 + 1), 1); add(4);
    if (c.tab.alloc(all.size() * sizeof(double2)) ||
        hipMemcpy(c.tab.p, all.data(), all.size() * sizeof(double2), hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipGetLastError();
        err = {E_NOMEM, "convolution table allocation failed"};
        return E_NOMEM;
    }
    const double2 *tab = (const double2 *)c.tab.p;
    c.Ff = mix_shape((int)P, rc, ntc, tab + at[0]);
    c.Fi = mix_shape((int)P, rci, ntc, tab + at[1]);
    c.Rf = mix_shape((int)M, rr, ntr, tab + at[2]);
    c.Ri = mix_shape((int)M, rr, ntr, tab + at[3]);
    c.rtw = tab + at[4];
    const size_t qp = (size_t)c.nblk << c.lcb;   // bins per row, whole blocks
    const size_t spec = (size_t)c.B * c.H * qp * sizeof(double2);
    if (c.sx.alloc(spec) || c.sg.alloc(spec) || c.sk.alloc((size_t)c.KH * qp * sizeof(double2)) ||
        c.kt.alloc(qp * c.P * sizeof(double2)) || c.acc.alloc((size_t)c.nchunk * qp * c.P * sizeof(double2))) {
        err = {E_NOMEM, "convolution workspace allocation failed"};
        return E_NOMEM;
    }
    static std::once_flag attr_once;
    std::call_once(attr_once, [] {
        for (const void *f :
             {(const void *)k_conv_cols<CC_SPECTRUM, 3>, (const void *)k_conv_cols<CC_SPECTRUM, 4>,
              (const void *)k_conv_cols<CC_CONV, 3>, (const void *)k_conv_cols<CC_CONV, 4>,
              (const void *)k_conv_cols<CC_GK, 3>, (const void *)k_conv_cols<CC_GK, 4>,
              (const void *)k_conv_cols<CC_GK_FINAL, 3>, (const void *)k_conv_cols<CC_GK_FINAL, 4>,
              (const void *)k_conv_rows<3>, (const void *)k_conv_rows<4>, (const void *)k_conv_rows_inv<3>,
              (const void *)k_conv_rows_inv<4>})
            if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024 - 2048) != hipSuccess)
                (void)hipGetLastError();
    });
    c.fused = true;
    return OK;
}

static ConvSpec conv_spec(const Conv2d &c, const DevBuf &b, int rows)
{
    return ConvSpec{(double2 *)b.p, rows, c.nblk, c.lcb};
}

// bytes from the first image of a workgroup's rows to the end of its last one
static long long conv_row_span(const Conv2d &c, const ConvSpec &S)
{
    const long long imgs = ((1 << c.ltb) + S.rows - 1) / S.rows + 1;
    return imgs * (((long long)S.nblk * S.rows) << S.lcb) * 16;
}

static size_t row_lds(const Conv2d &c) { return ((size_t)(c.Q / 2) << c.ltb) * sizeof(double2); }

// workgroups of up to 256 threads run faster with three waves per SIMD, larger ones with four (the
// rule of the engine's mixed-radix passes): forward of 21 x 439 x 1713, 13 x 9: 0.260 ms with four,
// 0.227 ms with three; of 16 x 2048^2, 63 x 63: 0.96 and 1.17 ms
static bool conv_w3(unsigned block) { return block <= 256; }

static ConvRowSet row_set(const Conv2d &c, const void *src, long long rows, int W, int rx, const ConvSpec &S)
{
    return ConvRowSet{src, S, rows, conv_row_span(c, S), W, rx, (unsigned)((rows + (1LL << c.ltb) - 1) >> c.ltb)};
}

static hipError_t rows_fwd(const Conv2d &c, std::initializer_list<ConvRowSet> sets, hipStream_t s)
{
    ConvRows R{};
    unsigned grid = 0;
    for (const ConvRowSet &a : sets) {
        R.set[R.nset++] = a;
        grid += a.groups;
    }
    R.F = c.Rf;
    R.rtw = c.rtw;
    R.f32 = c.dtype == 1;
    R.ltb = c.ltb;
    const unsigned block = (unsigned)c.Rf.NT << c.ltb;
    if (conv_w3(block)) hipLaunchKernelGGL(k_conv_rows<3>, dim3(grid), dim3(block), row_lds(c), s, R);
    else hipLaunchKernelGGL(k_conv_rows<4>, dim3(grid), dim3(block), row_lds(c), s, R);
    return hipGetLastError();
}

static ConvRowInvSet row_inv_set(const Conv2d &c, const ConvSpec &S, long long rows, void *dst, int Wout, int ox)
{
    return ConvRowInvSet{S, dst, rows, conv_row_span(c, S), Wout, ox, (unsigned)((rows + (1LL << c.ltb) - 1) >> c.ltb)};
}

static hipError_t rows_inv(const Conv2d &c, std::initializer_list<ConvRowInvSet> sets, hipStream_t s)
{
    ConvRowsInv R{};
    unsigned grid = 0;
    for (const ConvRowInvSet &a : sets)
        if (a.dst) {
            R.set[R.nset++] = a;
            grid += a.groups;
        }
    if (!grid) return hipSuccess;
    R.F = c.Ri;
    R.rtw = c.rtw;
    R.f32 = c.dtype == 1;
    R.ltb = c.ltb;
    R.scale = 1.0 / ((double)c.P * c.Q);
    const unsigned block = (unsigned)c.Ri.NT << c.ltb;
    if (conv_w3(block)) hipLaunchKernelGGL(k_conv_rows_inv<3>, dim3(grid), dim3(block), row_lds(c), s, R);
    else hipLaunchKernelGGL(k_conv_rows_inv<4>, dim3(grid), dim3(block), row_lds(c), s, R);
    return hipGetLastError();
}

template <int MODE>
static hipError_t cols(const Conv2d &c, ConvCols C, hipStream_t s)
{
    C.KT = (double2 *)c.kt.p;
    C.acc = (double2 *)c.acc.p;
    C.F = MODE == CC_GK_FINAL ? c.Fi : c.Ff;
    C.I = c.Fi;
    C.nchunk = c.nchunk;
    C.chunk = c.chunk;
    C.sub = c.sub;
    const unsigned cb = 1u << c.lcb, nblk = (unsigned)c.nblk;
    const unsigned ncol = MODE == CC_GK ? 2u * (unsigned)c.sub : cb;
    const unsigned grid = MODE == CC_CONV ? nblk * (unsigned)C.nimg
                          : MODE == CC_GK ? nblk * (cb / (unsigned)c.sub) * (unsigned)c.nchunk
                                          : nblk;
    const unsigned block = ncol * (unsigned)c.Ff.NT;
    const size_t lds = (size_t)ncol * (size_t)(c.P + 8) * sizeof(double2);
    if (conv_w3(block)) hipLaunchKernelGGL((k_conv_cols<MODE, 3>), dim3(grid), dim3(block), lds, s, C);
    else hipLaunchKernelGGL((k_conv_cols<MODE, 4>), dim3(grid), dim3(block), lds, s, C);
    return hipGetLastError();
}

static int conv_plan(std::unique_ptr<Plan> &p, int kind, int batch, long long P, long long Q, int forward, Error &err)
{
    const size_t shp3[3] = {(size_t)batch, (size_t)P, (size_t)Q};
    const long long Qh = Q / 2 + 1;
    // real side C-contiguous [B, P, Q]; complex side C-contiguous [B, P, Q/2+1]
    const ptrdiff_t sr[3] = {(ptrdiff_t)(P * Q * 8), (ptrdiff_t)(Q * 8), 8};
    const ptrdiff_t sc[3] = {(ptrdiff_t)(P * Qh * 16), (ptrdiff_t)(Qh * 16), 16};
    const size_t axes[2] = {1, 2};
    const bool real_in = (kind == 1 || kind == 4);
    return plan_create(p, kind, 0, 3, shp3, real_in ? sr : sc, real_in ? sc : sr, 2, axes, forward, err);
}

int conv2d_create(Conv2d **out, int B, int H, int W, int KH, int KW, int dtype, Error &err)
{
    if (B < 1 || H < 1 || W < 1 || KH < 1 || KW < 1 || KH > H || KW > W || (dtype != 0 && dtype != 1)) {
        err = {E_INVALID, "invalid convolution shape or dtype"};
        return E_INVALID;
    }
    auto c = std::make_unique<Conv2d>();
    c->B = B; c->H = H; c->W = W; c->KH = KH; c->KW = KW; c->dtype = dtype;
    c->P = conv_len((long long)H + KH - 1, false);
    c->Q = conv_len((long long)W + KW - 1, true);
    c->nspec = c->P * (c->Q / 2 + 1);
    int rc;
    if (conv_fused_setup(*c, err) != OK) return err.code;
    if (c->fused) {
        *out = c.release();
        return OK;
    }
    if ((rc = conv_plan(c->r2c_b, 1, B, c->P, c->Q, 1, err)) != OK) return rc;
    if ((rc = conv_plan(c->r2c_1, 1, 1, c->P, c->Q, 1, err)) != OK) return rc;
    if ((rc = conv_plan(c->c2r_b, 2, B, c->P, c->Q, 0, err)) != OK) return rc;
    if ((rc = conv_plan(c->c2r_adj_b, 4, B, c->P, c->Q, 0, err)) != OK) return rc;
    if ((rc = conv_plan(c->r2c_adj_b, 3, B, c->P, c->Q, 1, err)) != OK) return rc;
    if ((rc = conv_plan(c->r2c_adj_1, 3, 1, c->P, c->Q, 1, err)) != OK) return rc;
    const size_t real_b = (size_t)B * c->P * c->Q * 8, spec_b = (size_t)B * c->nspec * 16;
    if (c->pad.alloc(real_b) || c->spec_a.alloc(spec_b) || c->spec_b.alloc(spec_b) || c->kspec.alloc(c->nspec * 16) ||
        c->kpad.alloc((size_t)c->P * c->Q * 8)) {
        err = {E_NOMEM, "convolution workspace allocation failed"};
        return E_NOMEM;
    }
    *out = c.release();
    return OK;
}

static hipError_t pad(const Conv2d &c, const void *src, bool f32, double *dst, int B, int H, int W, int oy, int ox,
                      hipStream_t s)
{
    const unsigned g = blocks_for((long long)B * c.P * c.Q);
    if (f32) hipLaunchKernelGGL(k_pad2d<float>, dim3(g), dim3(256), 0, s, (const float *)src, dst, B, H, W, (int)c.P, (int)c.Q, oy, ox);
    else hipLaunchKernelGGL(k_pad2d<double>, dim3(g), dim3(256), 0, s, (const double *)src, dst, B, H, W, (int)c.P, (int)c.Q, oy, ox);
    return hipGetLastError();
}

static hipError_t crop(const Conv2d &c, const double *src, void *dst, bool f32, int B, int H, int W, int oy, int ox,
                       double scale, hipStream_t s)
{
    const unsigned g = blocks_for((long long)B * H * W);
    if (f32) hipLaunchKernelGGL(k_crop2d<float>, dim3(g), dim3(256), 0, s, src, (float *)dst, B, H, W, (int)c.P, (int)c.Q, oy, ox, scale);
    else hipLaunchKernelGGL(k_crop2d<double>, dim3(g), dim3(256), 0, s, src, (double *)dst, B, H, W, (int)c.P, (int)c.Q, oy, ox, scale);
    return hipGetLastError();
}

#define IFFT_TRY_HIP(expr)                                                                  \
    do {                                                                                    \
        hipError_t e_ = (expr);                                                             \
        if (e_ != hipSuccess) {                                                             \
            err = {E_HIP, std::string("convolution launch failed: ") + hipGetErrorString(e_)}; \
            return E_HIP;                                                                   \
        }                                                                                   \
    } while (0)
#define IFFT_TRY(expr)               \
    do {                             \
        int r_ = (expr);             \
        if (r_ != OK) return r_;     \
    } while (0)

// K^ = r2c(pad_0 k)
static int kernel_spectrum(Conv2d &c, const void *k, hipStream_t s, Error &err)
{
    IFFT_TRY_HIP(pad(c, k, c.dtype == 1, (double *)c.kpad.p, 1, c.KH, c.KW, 0, 0, s));
    return plan_execute(*c.r2c_1, c.kpad.p, c.kspec.p, 1.0, s, err);
}

// y = crop_c(c2r(K^ . r2c(pad_0 x))) / (P Q)
static int fused_forward(Conv2d &c, const void *x, const void *k, void *y, hipStream_t s, Error &err)
{
    const int cy = (c.KH - 1) / 2, cx = (c.KW - 1) / 2;
    const long long rows = (long long)c.B * c.H;
    const ConvSpec S = conv_spec(c, c.sx, c.H), Sk = conv_spec(c, c.sk, c.KH);
    IFFT_TRY_HIP(rows_fwd(c, {row_set(c, k, c.KH, c.KW, 0, Sk), row_set(c, x, rows, c.W, 0, S)}, s));
    ConvCols K{}, C{};
    K.Sa = Sk;
    IFFT_TRY_HIP(cols<CC_SPECTRUM>(c, K, s));
    C.Sa = C.So = S;   // in place: a workgroup reads its columns before it writes them
    C.oy = cy;
    C.nimg = c.B;
    IFFT_TRY_HIP(cols<CC_CONV>(c, C, s));
    IFFT_TRY_HIP(rows_inv(c, {row_inv_set(c, S, rows, y, c.W, cx)}, s));
    return OK;
}

// gx = crop_0(c2r(conj(K^) . G^)) / (P Q), gk = crop_0(c2r(sum_b conj(X^_b) . G^_b)) / (P Q),
// G^_b = r2c(pad_c g_b): the correlations that are the adjoints of the forward map
static int fused_backward(Conv2d &c, const void *x, const void *k, const void *gy, void *gx, void *gk, hipStream_t s,
                          Error &err)
{
    const int cy = (c.KH - 1) / 2, cx = (c.KW - 1) / 2;
    const long long rows = (long long)c.B * c.H;
    const ConvSpec Sx = conv_spec(c, c.sx, c.H), Sg = conv_spec(c, c.sg, c.H), Sk = conv_spec(c, c.sk, c.KH);
    const ConvRowSet rg = row_set(c, gy, rows, c.W, cx, Sg), rk = row_set(c, k, c.KH, c.KW, 0, Sk),
                     rx = row_set(c, x, rows, c.W, 0, Sx);
    if (gx && gk) IFFT_TRY_HIP(rows_fwd(c, {rk, rg, rx}, s));
    else if (gx) IFFT_TRY_HIP(rows_fwd(c, {rk, rg}, s));
    else if (gk) IFFT_TRY_HIP(rows_fwd(c, {rg, rx}, s));
    if (gx) {   // K^ before the kernel rows' workspace is reused
        ConvCols K{};
        K.Sa = Sk;
        IFFT_TRY_HIP(cols<CC_SPECTRUM>(c, K, s));
    }
    if (gk) {
        // sum_b conj(X^_b) G^_b per chunk of images, then the chunks' sum transformed back
        ConvCols C{};
        C.Sa = Sx;
        C.Sg = Sg;
        C.rg = cy;
        C.nimg = c.B;
        IFFT_TRY_HIP(cols<CC_GK>(c, C, s));
        ConvCols F{};
        F.Sa = F.So = Sk;
        IFFT_TRY_HIP(cols<CC_GK_FINAL>(c, F, s));
    }
    if (gx) {
        // the convolution pass with conj(K^), G^'s rows at cy, result rows from 0, in place
        ConvCols C{};
        C.Sa = C.So = Sg;
        C.ra = cy;
        C.nimg = c.B;
        C.conjk = 1;
        IFFT_TRY_HIP(cols<CC_CONV>(c, C, s));
    }
    IFFT_TRY_HIP(rows_inv(c, {row_inv_set(c, Sk, c.KH, gk, c.KW, 0), row_inv_set(c, Sg, rows, gx, c.W, 0)}, s));
    return OK;
}

int conv2d_forward(Conv2d &c, const void *x, const void *k, void *y, hipStream_t s, Error &err)
{
    if (c.fused) return fused_forward(c, x, k, y, s, err);
    const bool f32 = c.dtype == 1;
    IFFT_TRY(kernel_spectrum(c, k, s, err));
    IFFT_TRY_HIP(pad(c, x, f32, (double *)c.pad.p, c.B, c.H, c.W, 0, 0, s));
    IFFT_TRY(plan_execute(*c.r2c_b, c.pad.p, c.spec_a.p, 1.0, s, err));
    hipLaunchKernelGGL(k_spec_mul, dim3(blocks_for(c.B * c.nspec)), dim3(256), 0, s, (const double2 *)c.spec_a.p,
                       (const double2 *)c.kspec.p, (double2 *)c.spec_a.p, c.B, c.nspec, 0);
    IFFT_TRY_HIP(hipGetLastError());
    IFFT_TRY(plan_execute(*c.c2r_b, c.spec_a.p, c.pad.p, 1.0, s, err));
    const int cy = (c.KH - 1) / 2, cx = (c.KW - 1) / 2;
    IFFT_TRY_HIP(crop(c, (const double *)c.pad.p, y, f32, c.B, c.H, c.W, cy, cx, 1.0 / ((double)c.P * c.Q), s));
    return OK;
}

int conv2d_backward(Conv2d &c, const void *x, const void *k, const void *gy, void *gx, void *gk, hipStream_t s, Error &err)
{
    if (c.fused) return fused_backward(c, x, k, gy, gx, gk, s, err);
    const bool f32 = c.dtype == 1;
    const int cy = (c.KH - 1) / 2, cx = (c.KW - 1) / 2;
    const double inv = 1.0 / ((double)c.P * c.Q);
    IFFT_TRY(kernel_spectrum(c, k, s, err));
    // G_b = c2r*(pad_c g_b) / (P Q)
    IFFT_TRY_HIP(pad(c, gy, f32, (double *)c.pad.p, c.B, c.H, c.W, cy, cx, s));
    IFFT_TRY(plan_execute(*c.c2r_adj_b, c.pad.p, c.spec_b.p, inv, s, err));
    if (gk) {
        // X^_b recomputed, then sum_b conj(X^_b) G_b -> r2c* -> crop
        IFFT_TRY_HIP(pad(c, x, f32, (double *)c.pad.p, c.B, c.H, c.W, 0, 0, s));
        IFFT_TRY(plan_execute(*c.r2c_b, c.pad.p, c.spec_a.p, 1.0, s, err));
        hipLaunchKernelGGL(k_spec_corr_reduce, dim3(blocks_for(c.nspec)), dim3(256), 0, s, (const double2 *)c.spec_a.p,
                           (const double2 *)c.spec_b.p, (double2 *)c.spec_a.p, c.B, c.nspec);
        IFFT_TRY_HIP(hipGetLastError());
        IFFT_TRY(plan_execute(*c.r2c_adj_1, c.spec_a.p, c.kpad.p, 1.0, s, err));
        IFFT_TRY_HIP(crop(c, (const double *)c.kpad.p, gk, f32, 1, c.KH, c.KW, 0, 0, 1.0, s));
    }
    if (gx) {
        hipLaunchKernelGGL(k_spec_mul, dim3(blocks_for(c.B * c.nspec)), dim3(256), 0, s, (const double2 *)c.spec_b.p,
                           (const double2 *)c.kspec.p, (double2 *)c.spec_b.p, c.B, c.nspec, 1);
        IFFT_TRY_HIP(hipGetLastError());
        IFFT_TRY(plan_execute(*c.r2c_adj_b, c.spec_b.p, c.pad.p, 1.0, s, err));
        IFFT_TRY_HIP(crop(c, (const double *)c.pad.p, gx, f32, c.B, c.H, c.W, 0, 0, 1.0, s));
    }
    return OK;
}

void conv2d_grid(const Conv2d &c, long long &P, long long &Q) { P = c.P; Q = c.Q; }
void conv2d_destroy(Conv2d *c) { delete c; }

}  // namespace ifft
