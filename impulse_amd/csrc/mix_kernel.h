// The engine's mixed-radix pass kernel (mix_fft.h stages between the geometry
// of fft_params.h): one template per load and store mode, instantiated a few to
// a file (fft_mix*.hip) so that the files compile in parallel.
#pragma once

#include "mix_fft.h"

namespace ifft {

// ---------------------------------------------------------------------------
// load side: element `pos` of this thread's transform, byte offsets in 31 bits
// (checked at plan time)
// ---------------------------------------------------------------------------

template <int LM>
struct MixIn {
    const FftParams &P;
    __amdgpu_buffer_rsrc_t r;
    int es, ba, bb, step;     // element bytes, byte offset of element 0 of rows a / b, bytes per position
    int p0, dp;               // position of local point 0, positions per local point
    bool hasb;

    __device__ __forceinline__ MixIn(const FftParams &P_, const TfInfo &T) : P(P_)
    {
        r = make_rsrc((const char *)P.src + P.src_lo, P.src_span);
        constexpr bool cplx = LM == LD_C2C || LM == LD_C2R_HALF || LM == LD_C2R_PAIR;
        es = (cplx ? 16 : 8) >> P.src32;
        ba = (int)(T.ia * es - P.src_lo);
        bb = (int)(T.ib * es - P.src_lo);
        step = (int)P.in.sax * es;
        p0 = (int)T.ip0;
        dp = (int)P.in.pst;
        hasb = T.flags & 2;
    }

    // complex words at byte offsets o + q d
    template <int R> __device__ __forceinline__ void cload(double2 *v, int o, int d) const
    {
        if (P.src32) {
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const float2 f = bloadf2(r, o + q * d);
                v[q] = make_double2((double)f.x, (double)f.y);
            }
        } else {
#pragma unroll
            for (int q = 0; q < R; ++q) v[q] = bload2(r, o + q * d);
        }
    }
    // real words at byte offsets oa + q da (real part) and ob + q da (imaginary part)
    template <int R> __device__ __forceinline__ void rload(double2 *v, int oa, int ob, int d) const
    {
        if (P.src32) {
#pragma unroll
            for (int q = 0; q < R; ++q)
                v[q] = make_double2((double)bloadf1(r, oa + q * d), (double)bloadf1(r, ob + q * d));
        } else {
#pragma unroll
            for (int q = 0; q < R; ++q) v[q] = make_double2(bload1(r, oa + q * d), bload1(r, ob + q * d));
        }
    }

    template <int R> __device__ __forceinline__ void load(double2 *v, int b, int nb) const
    {
        const int pos = p0 + b * dp, dpos = nb * dp;
        if constexpr (LM == LD_C2C) {
            cload<R>(v, ba + pos * step, dpos * step);
        } else if constexpr (LM == LD_REAL_HALF) {
            if (P.in_words) cload<R>(v, ba + pos * 2 * step, dpos * 2 * step);
            else rload<R>(v, ba + pos * 2 * step, ba + pos * 2 * step + step, dpos * 2 * step);
        } else if constexpr (LM == LD_R2C_PAIR) {
            rload<R>(v, ba + pos * step, bb + pos * step, dpos * step);
            if (!hasb)
#pragma unroll
                for (int q = 0; q < R; ++q) v[q].y = 0.0;
        } else {
            static_assert(LM == LD_C2C, "a direct load mode");
        }
    }

    // Points k and M - k of a c2r signal, for k, k + d, ... (C of them, up to
    // `top`; the loads of all C are issued before the first product).
    //   half-length: z[k] = (X[k] + X*[M-k]) + i (X[k] - X*[M-k]) W_{2M}^{-k}; z[M-k] has the same
    //   sum and product conjugated
    //   odd pair: A[k] + i B[k] and conj(A[k]) + i conj(B[k])
    // Im of bin 0 (and of bin M of an even signal) is ignored; the adjoint halves all other bins.
    // put(k, z) takes the points.
    template <int C, class PUT> __device__ __forceinline__ void pairs(const PUT &put, int k0, int d, int top) const
    {
        const int M = P.M;
        double2 x[C], m[C], w[C];
        if constexpr (LM == LD_C2R_HALF) {
            const __amdgpu_buffer_rsrc_t rw = make_rsrc(P.rtw, ((long long)M + 1) * 16);
#pragma unroll
            for (int c = 0; c < C; ++c) w[c] = bload2(rw, min(k0 + c * d, top) * 16);
        }
        const int oa = ba, ob = LM == LD_C2R_HALF ? ba + M * step : bb, sb = LM == LD_C2R_HALF ? -step : step;
        if (P.src32) {
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int k = min(k0 + c * d, top);
                const float2 f = bloadf2(r, oa + k * step), g = bloadf2(r, ob + k * sb);
                x[c] = make_double2((double)f.x, (double)f.y);
                m[c] = make_double2((double)g.x, (double)g.y);
            }
        } else {
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int k = min(k0 + c * d, top);
                x[c] = bload2(r, oa + k * step);
                m[c] = bload2(r, ob + k * sb);
            }
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int k = k0 + c * d;
            if (k > top) break;
            double2 a = x[c], b = m[c];
            if (LM == LD_C2R_PAIR && !hasb) b = make_double2(0.0, 0.0);
            if (P.fwd_flag) { a = cconj(a); b = cconj(b); }
            if (k == 0) a.y = b.y = 0.0;
            else if (P.adj_w) { a = cscale(a, 0.5); b = cscale(b, 0.5); }
            if constexpr (LM == LD_C2R_HALF) {
                const double2 e = cadd(a, cconj(b));
                const double2 o = cmul(csub(a, cconj(b)), cconj(w[c]));
                put(k, make_double2(e.x - o.y, e.y + o.x));
                if (k && 2 * k != M) put(M - k, make_double2(e.x + o.y, o.x - e.y));
            } else {
                put(k, make_double2(a.x - b.y, a.y + b.x));
                if (k) put(M - k, make_double2(a.x + b.y, b.x - a.y));
            }
        }
    }
};

// ---------------------------------------------------------------------------
// store side
// ---------------------------------------------------------------------------

template <int SM>
struct MixOut {
    const FftParams &P;
    __amdgpu_buffer_rsrc_t r;
    int es, ba, bb, step;
    int p0, dp;
    long long j;
    bool hasb;

    __device__ __forceinline__ MixOut(const FftParams &P_, const TfInfo &T) : P(P_)
    {
        r = make_rsrc((char *)P.dst + P.dst_lo, P.dst_span);
        constexpr bool cplx = SM != ST_C2R_HALF && SM != ST_C2R_PAIR;
        es = (cplx ? 16 : 8) >> P.dst32;
        ba = (int)(T.oa * es - P.dst_lo);
        bb = (int)(T.ob * es - P.dst_lo);
        step = (int)P.out.sax * es;
        p0 = (int)T.op0;
        dp = (int)P.out.pst;
        j = T.j;
        hasb = T.flags & 4;
    }

    template <int R> __device__ __forceinline__ void cstore(const double2 *v, int o, int d, double f) const
    {
        if (P.dst32) {
#pragma unroll
            for (int q = 0; q < R; ++q) bstoref2(r, o + q * d, cscale(v[q], f));
        } else {
#pragma unroll
            for (int q = 0; q < R; ++q) bstore2(r, o + q * d, cscale(v[q], f));
        }
    }
    template <int R> __device__ __forceinline__ void rstore(const double2 *v, int oa, int ob, int d, bool both) const
    {
        const double f = P.fct;
        if (P.dst32) {
#pragma unroll
            for (int q = 0; q < R; ++q) {
                bstoref1(r, oa + q * d, v[q].x * f);
                if (both) bstoref1(r, ob + q * d, v[q].y * f);
            }
        } else {
#pragma unroll
            for (int q = 0; q < R; ++q) {
                bstore1(r, oa + q * d, v[q].x * f);
                if (both) bstore1(r, ob + q * d, v[q].y * f);
            }
        }
    }
    __device__ __forceinline__ void c1(int o, double2 z) const
    {
        if (P.dst32) bstoref2(r, o, z);
        else bstore2(r, o, z);
    }

    template <int R, class G> __device__ __forceinline__ void store(const double2 *v, int n, int dn, G) const
    {
        const int pos = p0 + n * dp, dpos = dn * dp;
        if constexpr (SM == ST_C2C) {
            cstore<R>(v, ba + pos * step, dpos * step, P.fct);
        } else if constexpr (SM == ST_TWIDDLE) {
            const long long S = 1LL << P.tw_logS;
            const __amdgpu_buffer_rsrc_t rlo = make_rsrc(P.tw_lo, S * 16);
            const __amdgpu_buffer_rsrc_t rhi = make_rsrc(P.tw_hi, (P.tw_L / S + 2) * 16);
            const double s = (double)P.sign;
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const double2 w = twolevel_b(rlo, rhi, P.tw_logS, j * (long long)(n + q * dn));
                bstore2(r, ba + (pos + q * dpos) * step, cmul(v[q], tw_sign(w, s)));
                if (q % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // four twiddles in flight, not R
            }
        } else if constexpr (SM == ST_C2R_HALF) {
            if (P.out_words) cstore<R>(v, ba + pos * 2 * step, dpos * 2 * step, P.fct);
            else rstore<R>(v, ba + pos * 2 * step, ba + pos * 2 * step + step, dpos * 2 * step, true);
        } else {
            static_assert(SM == ST_C2R_PAIR, "a direct store mode");
            rstore<R>(v, ba + pos * step, bb + pos * step, dpos * step, hasb);
        }
    }

    // bins k and M - k of an even real transform from Z[k], Z[M - k] (W = W_{2M}^k)
    __device__ __forceinline__ void half_pair(int k, double2 zk, double2 zm, double2 w) const
    {
        const int M = P.M, km = M - k;
        const double2 e1 = cscale(cadd(zk, cconj(zm)), 0.5), d1 = csub(zk, cconj(zm));
        const double2 o1 = make_double2(0.5 * d1.y, -0.5 * d1.x);
        const double2 e2 = cscale(cadd(zm, cconj(zk)), 0.5), d2 = csub(zm, cconj(zk));
        const double2 o2 = make_double2(0.5 * d2.y, -0.5 * d2.x);
        const double f1 = (P.adj_w && k != 0) ? 2.0 * P.fct : P.fct;
        double2 a = cscale(cadd(e1, cmul(o1, w)), f1);
        double2 b = cscale(cadd(e2, cmul(o2, make_double2(-w.x, w.y))), f1);
        if (!P.fwd_flag) { a = cconj(a); b = cconj(b); }
        c1(ba + k * step, a);
        if (km != k) c1(ba + km * step, b);
    }
    // bin k of both rows of an odd pair from Z[k], Z[L - k]
    __device__ __forceinline__ void odd_pair(int k, double2 zk, double2 zl) const
    {
        const double2 zm = cconj(zl), d = csub(zk, zm);
        const double f = (P.adj_w && k != 0) ? 2.0 * P.fct : P.fct;
        double2 xa = cscale(cadd(zk, zm), 0.5 * f);
        double2 xb = make_double2(0.5 * f * d.y, -0.5 * f * d.x);
        if (!P.fwd_flag) { xa = cconj(xa); xb = cconj(xb); }
        c1(ba + k * step, xa);
        if (hasb) c1(bb + k * step, xb);
    }
};

// the half spectra of a real transform from its points in the LDS row
template <int SM>
__device__ __forceinline__ void mix_real_out(const FftParams &P, const TfInfo &T, const double2 *row, int i, int NT)
{
    const MixOut<SM> out(P, T);
    const int M = P.M;
    if constexpr (SM == ST_R2C_HALF) {
        for (int k = i; 2 * k <= M; k += NT) out.half_pair(k, row[k], row[k ? M - k : 0], P.rtw[k]);
    } else {
        for (int k = i; 2 * k <= M; k += NT) out.odd_pair(k, row[k], row[k ? M - k : 0]);
    }
}

template <int LM, int SM, int WPE>
__global__ void __launch_bounds__(kMixMaxThreads) __attribute__((amdgpu_waves_per_eu(WPE)))
k_fft_mix(const FftParams P)
{
    extern __shared__ double2 lds[];
    __shared__ TfInfo info[kMaxTB];
    constexpr bool LD_LDS = LM == LD_C2R_HALF || LM == LD_C2R_PAIR;
    constexpr bool ST_LDS = SM == ST_R2C_HALF || SM == ST_R2C_PAIR;
    const int tid = (int)threadIdx.x, TB = P.TB, NT = P.NT;
    const long long g0 = (long long)xcd_block(blockIdx.x, gridDim.x) * TB;
    if (tid < TB) info[tid] = make_tfinfo(P, g0 + tid);
    const int tl = P.col_load ? tid % TB : tid / NT, il = P.col_load ? tid / TB : tid % NT;
    const int ts = P.col_store ? tid % TB : tid / NT, is = P.col_store ? tid / TB : tid % NT;
    __syncthreads();
    MixShape S;
    S.N = P.N;
    S.nst = P.nst;
    S.codes = P.codes;
    S.NT = NT;
    S.tw = P.tw;
    const MixIn<LM> in(P, info[tl]);
    const bool vin = info[tl].flags & 1, vout = info[ts].flags & 1;
    double2 *bl = lds + tl * P.LD, *bs = lds + ts * P.LD;
    const double s = (double)P.sign;
    auto stages = [&](const auto &st) __attribute__((always_inline)) {
        if constexpr (LD_LDS) {
            // the pre-processed points of a c2r signal come in pairs from one bin pair, so they are
            // staged through the LDS row; every bin is read once
            if (vin) {
                // four bin pairs in flight per thread
                const int top = LM == LD_C2R_HALF ? P.M / 2 : (P.M - 1) / 2;
                for (int k = il; k <= top; k += 4 * NT) in.template pairs<4>([&](int n, double2 z) { bl[n] = z; }, k, NT, top);
            }
            __syncthreads();
            mix_fft<true, ST_LDS>(S, MixLds{bl}, il, true, MixLds{bs}, is, vout, s, MixLds{bl}, st);
        } else {
            mix_fft<false, ST_LDS>(S, MixLds{bl}, il, vin, MixLds{bs}, is, vout, s, in, st);
        }
    };
    if constexpr (!ST_LDS) {
        stages(MixOut<SM>(P, info[ts]));
    } else {
        stages(MixLds{bs});
        if (vout) mix_real_out<SM>(P, info[ts], bs, is, NT);
    }
}

template <int LM, int SM, int WPE>
static hipError_t launch_mix_wpe(const FftParams &P, unsigned grid, unsigned block, size_t lds, hipStream_t s)
{
    static bool attr_done = false;
    if (!attr_done) {
        if (hipFuncSetAttribute((const void *)k_fft_mix<LM, SM, WPE>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                160 * 1024 - (int)(sizeof(TfInfo) * kMaxTB) - 1024) != hipSuccess)
            (void)hipGetLastError();
        attr_done = true;
    }
    hipLaunchKernelGGL((k_fft_mix<LM, SM, WPE>), dim3(grid), dim3(block), lds, s, P);
    return hipGetLastError();
}

template <int LM, int SM>
static hipError_t launch_mix(const FftParams &P, unsigned grid, unsigned block, size_t lds, hipStream_t s)
{
    return mix_wpe(grid, block) == 3 ? launch_mix_wpe<LM, SM, 3>(P, grid, block, lds, s)
                                     : launch_mix_wpe<LM, SM, 4>(P, grid, block, lds, s);
}

// ---------------------------------------------------------------------------
// Bluestein lengths in one pass: signal times the chirp, padded transform, product with the chirp
// kernel's spectrum, transform back, times the chirp (mix_conv: the product sits in registers)
//
// Against k_fft_lds with the same convolution (one call per stage, every point staged at both ends),
// on one MI355X: c2c rows 4096 x 1021 0.193 -> 0.082 ms, 50000 x 101 0.314 -> 0.065 ms, columns 1021 x
// 4096 0.223 -> 0.133 ms, r2c rows of 1021 0.099 -> 0.050 ms.  Two transforms of 2.1 times the length:
// bound by their LDS exchanges and the LDS rows' share of the CU, not by HBM.
// ---------------------------------------------------------------------------

// offset that no window reaches (spans are checked to end below it): loads give zero without touching
// memory, stores are dropped
constexpr int kMixNowhere = 0x7ffffff0;

template <int LM>
struct BlueIn {
    const MixIn<LM> in;
    const __amdgpu_buffer_rsrc_t rc;   // the chirp, P.M entries: zero beyond the signal
    const int Ls;
    const double cj;
    __device__ __forceinline__ BlueIn(const FftParams &P, const TfInfo &T)
        : in(P, T), rc(make_rsrc(P.chirp, (long long)P.M * 16)), Ls(P.M), cj(P.conj_in ? -1.0 : 1.0)
    {
    }
    template <int R> __device__ __forceinline__ void load(double2 *v, int b, int nb) const
    {
        const FftParams &P = in.P;
        if constexpr (LM == LD_C2C) {
            if (P.src32) {
#pragma unroll
                for (int q = 0; q < R; ++q) {
                    const float2 f = bloadf2(in.r, at(b + q * nb, in.ba, in.step));
                    v[q] = make_double2((double)f.x, (double)f.y);
                }
            } else {
#pragma unroll
                for (int q = 0; q < R; ++q) v[q] = bload2(in.r, at(b + q * nb, in.ba, in.step));
            }
        } else if constexpr (LM == LD_REAL_HALF) {
            if (P.in_words) {
                if (P.src32) {
#pragma unroll
                    for (int q = 0; q < R; ++q) {
                        const float2 f = bloadf2(in.r, at(b + q * nb, in.ba, 2 * in.step));
                        v[q] = make_double2((double)f.x, (double)f.y);
                    }
                } else {
#pragma unroll
                    for (int q = 0; q < R; ++q) v[q] = bload2(in.r, at(b + q * nb, in.ba, 2 * in.step));
                }
            } else {
#pragma unroll
                for (int q = 0; q < R; ++q)
                    v[q] = make_double2(real(at(b + q * nb, in.ba, 2 * in.step)),
                                        real(at(b + q * nb, in.ba + in.step, 2 * in.step)));
            }
        } else {
            static_assert(LM == LD_R2C_PAIR, "a direct load mode");
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const double a = real(at(b + q * nb, in.ba, in.step)), c = real(at(b + q * nb, in.bb, in.step));
                v[q] = make_double2(a, in.hasb ? c : 0.0);
            }
        }
#pragma unroll
        for (int q = 0; q < R; ++q) v[q] = chirped(v[q], b + q * nb);
    }
    __device__ __forceinline__ double2 chirped(double2 z, int pos) const
    {
        z.y *= cj;
        return cmul(z, bload2(rc, pos * 16));
    }
    __device__ __forceinline__ int at(int pos, int base, int step) const { return pos < Ls ? base + pos * step : kMixNowhere; }
    __device__ __forceinline__ double real(int o) const { return in.P.src32 ? (double)bloadf1(in.r, o) : bload1(in.r, o); }
};

struct BlueMul {
    __amdgpu_buffer_rsrc_t r;
    template <int R> __device__ __forceinline__ void apply(double2 *v, int b, int nb) const
    {
#pragma unroll
        for (int q = 0; q < R; ++q) v[q] = cmul(v[q], bload2(r, (b + q * nb) * 16));
    }
};

// outputs up to the signal's length times the chirp: to memory, or (real transforms) to the LDS row
template <int SM>
struct BlueOut {
    const MixOut<SM> out;
    const __amdgpu_buffer_rsrc_t rc;
    const int Ls;
    const double cj;
    double2 *row;
    __device__ __forceinline__ BlueOut(const FftParams &P, const TfInfo &T, double2 *row_)
        : out(P, T), rc(make_rsrc(P.chirp, (long long)P.M * 16)), Ls(P.M), cj(P.conj_out ? -1.0 : 1.0), row(row_)
    {
    }
    template <int R, class G> __device__ __forceinline__ void store(const double2 *v, int n, int dn, G) const
    {
        const FftParams &P = out.P;
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const int pos = n + q * dn;
            const bool ok = pos < Ls;
            double2 z = cmul(v[q], bload2(rc, pos * 16));
            z.y *= cj;
            if constexpr (SM == ST_R2C_HALF || SM == ST_R2C_PAIR) {
                if (ok) row[pos] = z;
            } else {
                z = cscale(z, P.fct);
                if constexpr (SM == ST_C2C) {
                    out.c1(ok ? out.ba + pos * out.step : kMixNowhere, z);
                } else if constexpr (SM == ST_C2R_HALF) {
                    const int o = ok ? out.ba + pos * 2 * out.step : kMixNowhere;
                    if (P.out_words) {
                        out.c1(o, z);
                    } else {
                        real(o, z.x);
                        real(ok ? o + out.step : kMixNowhere, z.y);
                    }
                } else {
                    real(ok ? out.ba + pos * out.step : kMixNowhere, z.x);
                    real(ok && out.hasb ? out.bb + pos * out.step : kMixNowhere, z.y);
                }
            }
        }
    }
    __device__ __forceinline__ void real(int o, double x) const
    {
        if (out.P.dst32) bstoref1(out.r, o, x);
        else bstore1(out.r, o, x);
    }
};

// idle slots of the last workgroup neither load nor store
template <int LM>
struct BlueGateIn {
    const BlueIn<LM> in;
    const bool valid;
    template <int R> __device__ __forceinline__ void load(double2 *v, int b, int nb) const
    {
        if (valid) in.template load<R>(v, b, nb);
    }
};
template <int SM>
struct BlueGate {
    const BlueOut<SM> &out;
    const bool valid;
    template <int R, class G> __device__ __forceinline__ void store(const double2 *v, int n, int dn, G g) const
    {
        if (valid) out.template store<R>(v, n, dn, g);
    }
};

template <int LM, int SM, int WPE>
__global__ void __launch_bounds__(kMixMaxThreads) __attribute__((amdgpu_waves_per_eu(WPE)))
k_fft_mix_blue(const FftParams P)
{
    extern __shared__ double2 lds[];
    __shared__ TfInfo info[kMaxTB];
    constexpr bool LD_LDS = LM == LD_C2R_HALF || LM == LD_C2R_PAIR;
    constexpr bool ST_LDS = SM == ST_R2C_HALF || SM == ST_R2C_PAIR;
    const int tid = (int)threadIdx.x, TB = P.TB, NT = P.NT, N = P.N;
    const long long g0 = (long long)xcd_block(blockIdx.x, gridDim.x) * TB;
    if (tid < TB) info[tid] = make_tfinfo(P, g0 + tid);
    const bool col = P.col_load || P.col_store;   // one mapping for both sides
    const int t = col ? tid % TB : tid / NT, i = col ? tid / TB : tid % NT;
    __syncthreads();
    MixShape F{N, P.nst, P.codes, NT, P.tw}, I{N, P.nst, P.codes_inv, NT, P.tw_inv};
    const TfInfo T = info[t];
    const bool valid = T.flags & 1;
    double2 *row = lds + t * P.LD;
    const BlueMul mul{make_rsrc(P.spec, (long long)N * 16)};
    const BlueOut<SM> out(P, T, row);
    if constexpr (LD_LDS) {
        const MixIn<LM> in(P, T);
        const __amdgpu_buffer_rsrc_t rc = make_rsrc(P.chirp, (long long)P.M * 16);
        const double cj = P.conj_in ? -1.0 : 1.0;
        auto put = [&](int n, double2 z) {
            z.y *= cj;
            row[n] = cmul(z, bload2(rc, n * 16));
        };
        const int top = LM == LD_C2R_HALF ? P.M / 2 : (P.M - 1) / 2;
        if (valid)
            for (int k = i; k <= top; k += 2 * NT) in.template pairs<2>(put, k, NT, top);
        for (int n = P.M + i; n < N; n += NT) row[n] = make_double2(0.0, 0.0);
        __syncthreads();
        mix_conv<true, ST_LDS>(F, I, row, i, MixLds{row}, mul, BlueGate<SM>{out, valid});
    } else {
        mix_conv<false, ST_LDS>(F, I, row, i, BlueGateIn<LM>{BlueIn<LM>(P, T), valid}, mul, BlueGate<SM>{out, valid});
    }
    if constexpr (ST_LDS)
        if (valid) mix_real_out<SM>(P, T, row, i, NT);
}

template <int LM, int SM, int WPE>
static hipError_t launch_mix_blue_wpe(const FftParams &P, unsigned grid, unsigned block, size_t lds, hipStream_t s)
{
    static bool attr_done = false;
    if (!attr_done) {
        if (hipFuncSetAttribute((const void *)k_fft_mix_blue<LM, SM, WPE>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                160 * 1024 - (int)(sizeof(TfInfo) * kMaxTB) - 1024) != hipSuccess)
            (void)hipGetLastError();
        attr_done = true;
    }
    hipLaunchKernelGGL((k_fft_mix_blue<LM, SM, WPE>), dim3(grid), dim3(block), lds, s, P);
    return hipGetLastError();
}

template <int LM, int SM>
static hipError_t launch_mix_blue(const FftParams &P, unsigned grid, unsigned block, size_t lds, hipStream_t s)
{
    return mix_wpe(grid, block) == 3 ? launch_mix_blue_wpe<LM, SM, 3>(P, grid, block, lds, s)
                                     : launch_mix_blue_wpe<LM, SM, 4>(P, grid, block, lds, s);
}

}  // namespace ifft
