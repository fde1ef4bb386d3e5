// Mixed-radix Stockham stages of runtime length, staged through LDS, with the
// first stage's inputs and the last stage's outputs going straight between
// registers and the caller's loads and stores.
//
// A length N = R0 R1 ... (two to four stages mostly, six at most, radices 2..16) is factored on the
// host (mix_factor).  Stage s of radix R, with p the product of the earlier
// radices, takes butterflies b in [0, N/R), k = b mod p:
//   inputs  x[b + q N/R] W_{pR}^{q k},  outputs y[(b - k) R + k + q p],  q < R,
// so the last stage (p = N/R) leaves y[b + q N/R] in natural order.  The
// composite radices 6, 10, 12, 14 and 15 are prime-factor products (index maps,
// no inner twiddles), 9 is 3 x 3.
//
// Against a kernel that stages every point through LDS before the first and
// after the last radix this halves the LDS round trips (two exchanges for a
// length up to 4096), and large composite radices keep that count low for
// lengths with no power of two in them.  Twiddles come from a table laid out in
// stage order (mix_table): the lanes of a wave read consecutive entries, and
// every twiddle is one rounding away from exact.
#pragma once

#include <type_traits>
#include <utility>

#include "butterflies.h"
#include "fft_common.h"

namespace ifft {

// ---------------------------------------------------------------------------
// composite butterflies
// ---------------------------------------------------------------------------

template <int R> __device__ __forceinline__ void dftm(double2 *v, double s);

// inverse of a modulo m (compile time)
__host__ __device__ constexpr int mod_inv(int a, int m)
{
    for (int x = 1; x < m; ++x)
        if (a * x % m == 1) return x;
    return 1;
}

// Prime-factor DFT of A B points (A, B coprime): input (B a + A b) mod N is
// point (a, b); output (ka, kb) is index k with k = ka mod A and k = kb mod B.
template <int A, int B>
__device__ __forceinline__ void dft_pfa(double2 *v, double s)
{
    constexpr int N = A * B;
    constexpr int EA = B * mod_inv(B % A, A), EB = A * mod_inv(A % B, B);
    double2 t[B][A];
#pragma unroll
    for (int b = 0; b < B; ++b) {
#pragma unroll
        for (int a = 0; a < A; ++a) t[b][a] = v[(B * a + A * b) % N];
        dftm<A>(t[b], s);
    }
#pragma unroll
    for (int a = 0; a < A; ++a) {
        double2 u[B];
#pragma unroll
        for (int b = 0; b < B; ++b) u[b] = t[b][a];
        dftm<B>(u, s);
#pragma unroll
        for (int b = 0; b < B; ++b) v[(EA * a + EB * b) % N] = u[b];
    }
}

// cos and sin of 2 pi k / 9, k = 1, 2, 4
__device__ __forceinline__ void dft9(double2 *v, double s)
{
    constexpr double c1 = 0.766044443118978, s1 = 0.6427876096865394;
    constexpr double c2 = 0.17364817766693036, s2 = 0.984807753012208;
    constexpr double c4 = -0.9396926207859084, s4 = 0.3420201433256687;
    double2 t[3][3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
#pragma unroll
        for (int m = 0; m < 3; ++m) t[j][m] = v[j + 3 * m];
        dft<3>(t[j], s);
    }
    t[1][1] = cmul(t[1][1], make_double2(c1, s * s1));
    t[1][2] = cmul(t[1][2], make_double2(c2, s * s2));
    t[2][1] = cmul(t[2][1], make_double2(c2, s * s2));
    t[2][2] = cmul(t[2][2], make_double2(c4, s * s4));
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        double2 u[3] = {t[0][k], t[1][k], t[2][k]};
        dft<3>(u, s);
#pragma unroll
        for (int m = 0; m < 3; ++m) v[k + 3 * m] = u[m];
    }
}

template <int R> __device__ __forceinline__ void dftm(double2 *v, double s)
{
    if constexpr (R == 6) dft_pfa<3, 2>(v, s);
    else if constexpr (R == 9) dft9(v, s);
    else if constexpr (R == 10) dft_pfa<5, 2>(v, s);
    else if constexpr (R == 12) dft_pfa<4, 3>(v, s);
    else if constexpr (R == 14) dft_pfa<7, 2>(v, s);
    else if constexpr (R == 15) dft_pfa<5, 3>(v, s);
    else dft<R>(v, s);
}

// ---------------------------------------------------------------------------
// stages
// ---------------------------------------------------------------------------

constexpr int kMixMaxStages = 6;

// f(std::integral_constant<int, 0>{}), ..., f(std::integral_constant<int, N - 1>{})
template <int N, class F, int... I>
__device__ __forceinline__ void each_of(F &&f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F> __device__ __forceinline__ void each(F &&f)
{
    each_of<N>(f, std::make_integer_sequence<int, N>{});
}

// butterflies of radix R a thread may own (16 points in registers at most)
__host__ __device__ constexpr int mix_nb(int R) { return R > 8 ? 1 : 16 / R; }

// The same value, untraceable for the compiler: everything a stage derives from the thread's slot,
// the length and the sign (addresses, products with the butterflies' constants) would otherwise be
// hoisted out of the stage loop for all fifteen radices at once, 180 registers more than there are.
__device__ __forceinline__ double opaque(double s)
{
    asm volatile("" : "+v"(s));
    return s;
}
__device__ __forceinline__ int opaque(int i)
{
    asm volatile("" : "+v"(i));
    return i;
}
__device__ __forceinline__ int opaque_scalar(int i) { return __builtin_amdgcn_readfirstlane(opaque(i)); }

// calls f(std::integral_constant<int, R>) for the runtime radix r (2..16), a uniform branch
template <class F>
__device__ __forceinline__ void mix_radix(int r, F &&f)
{
    switch (r) {
        case 2: f(std::integral_constant<int, 2>{}); break;
        case 3: f(std::integral_constant<int, 3>{}); break;
        case 4: f(std::integral_constant<int, 4>{}); break;
        case 5: f(std::integral_constant<int, 5>{}); break;
        case 6: f(std::integral_constant<int, 6>{}); break;
        case 7: f(std::integral_constant<int, 7>{}); break;
        case 8: f(std::integral_constant<int, 8>{}); break;
        case 9: f(std::integral_constant<int, 9>{}); break;
        case 10: f(std::integral_constant<int, 10>{}); break;
        case 11: f(std::integral_constant<int, 11>{}); break;
        case 12: f(std::integral_constant<int, 12>{}); break;
        case 13: f(std::integral_constant<int, 13>{}); break;
        case 14: f(std::integral_constant<int, 14>{}); break;
        case 15: f(std::integral_constant<int, 15>{}); break;
        default: f(std::integral_constant<int, 16>{}); break;
    }
}

// LDS end of a stage: point idx at buf[idx]
struct MixLds {
    double2 *buf;
    __device__ __forceinline__ double2 &at(int idx) const { return buf[idx]; }
    __device__ __forceinline__ double &word(int d) const { return ((double *)buf)[d]; }   // real view
    template <int R> __device__ __forceinline__ void load(double2 *v, int b, int nb) const
    {
#pragma unroll
        for (int q = 0; q < R; ++q) v[q] = buf[b + q * nb];
    }
    template <int R, class G> __device__ __forceinline__ void store(const double2 *v, int j, int p, G) const
    {
#pragma unroll
        for (int q = 0; q < R; ++q) buf[j + q * p] = v[q];
    }
};

// The same with one word skipped every 16, for lengths with no odd radix to put first: the first
// stage's writes, whose stride is the radix, then spread over the banks.
struct MixLdsPad {
    double2 *buf;
    static constexpr __host__ __device__ int pad(int idx) { return idx + (idx >> 4); }
    __device__ __forceinline__ double2 &at(int idx) const { return buf[pad(idx)]; }
    __device__ __forceinline__ double &word(int d) const { return ((double *)(buf + pad(d >> 1)))[d & 1]; }
    template <int R> __device__ __forceinline__ void load(double2 *v, int b, int nb) const
    {
#pragma unroll
        for (int q = 0; q < R; ++q) v[q] = buf[pad(b + q * nb)];
    }
    template <int R, class G> __device__ __forceinline__ void store(const double2 *v, int j, int p, G) const
    {
#pragma unroll
        for (int q = 0; q < R; ++q) buf[pad(j + q * p)] = v[q];
    }
};

// One stage: `ld` delivers inputs b, b + nb, ..., `st` takes outputs j, j + p, ... (and the number of
// the butterfly within the thread).
// SYNC separates the reads from the writes when both ends are the same LDS
// rows.  lim is the number of butterflies this thread's transform runs (N / R,
// or 0 for an idle slot).  Twiddle W_{pR}^{qk} sits at tw[(q - 1) p + k].  SG is
// the sign of the transform where it is known at compile time, else 0 and in s.
template <int R, bool FIRST, bool SYNC, int SG = 0, class LD, class ST>
__device__ __forceinline__ void mix_stage(int nb, int lim, int p, int i, int NT, double s, const double2 *tw,
                                          const LD &ld, const ST &st)
{
    constexpr int G = mix_nb(R);
    double2 v[G][R];
    s = SG ? (double)SG : opaque(s);
    i = opaque(i);
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int b = i + g * NT;
        if (b < lim) ld.template load<R>(v[g], b, nb);
    }
    if constexpr (SYNC) __syncthreads();
    const float rp = FIRST ? 1.0f : __builtin_amdgcn_rcpf((float)p);
    const __amdgpu_buffer_rsrc_t rtw = make_rsrc(tw, FIRST ? 0 : (long long)(R - 1) * p * 16);
    each<G>([&](auto gc) __attribute__((always_inline)) {
        constexpr int g = decltype(gc)::value;
        const int b = i + g * NT;
        if (b < lim) {
            const int k = FIRST ? 0 : mod_small(b, p, rp);
            if constexpr (!FIRST) {
#pragma unroll
                for (int q = 1; q < R; ++q) v[g][q] = cmul(v[g][q], bload2(rtw, (k + (q - 1) * p) * 16));
            }
            dftm<R>(v[g], s);
            st.template store<R>(v[g], (b - k) * R + k, p, gc);
        }
    });
}

// Radices of a length and its stage-ordered twiddle table, as kernels take them
struct MixShape {
    int N, nst;
    unsigned codes;      // radix - 1 of stage k in bits 4k .. 4k + 3
    int NT;              // threads per transform
    const double2 *tw;   // stage 1's table, then stage 2's, ... (sign of the transform)
};

// A whole transform: `ld` is the source of the first stage, `st` the
// destination of the last one (or the LDS rows themselves), `row` this thread's
// LDS row.  (i, on_in) and (o, orow, on_out) are the thread's slot on the load
// and store side, which may differ when lanes walk another way there.
// LD_LDS: the inputs already sit in the LDS rows (behind a barrier).  ST_LDS: the
// outputs stay in LDS rows, natural order; a barrier follows.
template <bool LD_LDS, bool ST_LDS, int SG = 0, class ROW, class LD, class ST>
__device__ __forceinline__ void mix_fft(const MixShape &S, const ROW &row, int i, bool on_in, const ROW &orow, int o,
                                        bool on_out, double s, const LD &ld, const ST &st)
{
    const int N = S.N, NT = S.NT;
    unsigned codes = S.codes;
    mix_radix((int)(codes & 15u) + 1, [&](auto rc) __attribute__((always_inline)) {
        constexpr int R = decltype(rc)::value;
        const int nb = opaque_scalar(N) / R;
        mix_stage<R, true, LD_LDS, SG>(nb, on_in ? nb : 0, 1, i, NT, s, nullptr, ld, row);
    });
    __syncthreads();
    int p = (int)(codes & 15u) + 1;
    const double2 *tw = S.tw;
    const int mid = ST_LDS ? S.nst : S.nst - 1;
    for (int k = 1; k < mid; ++k) {
        codes >>= 4;
        const int r = (int)(codes & 15u) + 1;
        mix_radix(r, [&](auto rc) __attribute__((always_inline)) {
            constexpr int R = decltype(rc)::value;
            const int nb = opaque_scalar(N) / R;
            mix_stage<R, false, true, SG>(nb, nb, p, i, NT, s, tw, row, row);
        });
        __syncthreads();
        tw += (r - 1) * p;
        p *= r;
    }
    if constexpr (!ST_LDS) {
        codes >>= 4;
        mix_radix((int)(codes & 15u) + 1, [&](auto rc) __attribute__((always_inline)) {
            constexpr int R = decltype(rc)::value;
            const int nb = N / R;
            mix_stage<R, false, false, SG>(nb, on_out ? nb : 0, p, o, NT, s, tw, orow, st);
        });
    }
}

// The turn of mix_conv: the forward outputs of a butterfly times `mul`'s values, and the first
// inverse stage (outputs b R + q) into the LDS row.
template <class MUL>
struct MixTurn {
    const MixLds &row;
    const MUL &mul;
    template <int R, class G> __device__ __forceinline__ void store(double2 *v, int b, int nb, G g) const
    {
        mul.template apply<R>(v, b, nb);
        dftm<R>(v, 1.0);
        row.template store<R>(v, b * R, 1, g);
    }
};

// Forward transform, pointwise product and inverse transform of one LDS row.  The inverse takes the
// forward radices in reverse, so its first stage has its inputs b + q N/R where the forward's last
// stage leaves its outputs: that radix is transformed, multiplied (mul) and transformed back in
// registers, and the spectrum never passes through LDS.  F: forward shape (sign -1 table), I: the
// reversed one (sign +1 table), of the same threads.
// LD_LDS / ST_LDS as for mix_fft.
template <bool LD_LDS = false, bool ST_LDS = false, class LD, class MUL, class ST>
__device__ __forceinline__ void mix_conv(const MixShape &F, const MixShape &I, double2 *buf, int i, const LD &ld,
                                         const MUL &mul, const ST &st)
{
    const int N = F.N, NT = F.NT;
    const MixLds row{buf};
    unsigned codes = F.codes;
    mix_radix((int)(codes & 15u) + 1, [&](auto rc) __attribute__((always_inline)) {
        constexpr int R = decltype(rc)::value;
        const int nb = N / R;
        mix_stage<R, true, LD_LDS, -1>(nb, nb, 1, i, NT, -1.0, nullptr, ld, row);
    });
    __syncthreads();
    int p = (int)(codes & 15u) + 1;
    const double2 *tw = F.tw;
    auto middle = [&](auto sg) __attribute__((always_inline)) {
        constexpr int SG = decltype(sg)::value;
        for (int k = 1; k < F.nst - 1; ++k) {
            codes >>= 4;
            const int r = (int)(codes & 15u) + 1;
            mix_radix(r, [&](auto rc) __attribute__((always_inline)) {
                constexpr int R = decltype(rc)::value;
                const int nb = opaque_scalar(N) / R;
                mix_stage<R, false, true, SG>(nb, nb, p, i, NT, (double)SG, tw, row, row);
            });
            __syncthreads();
            tw += (r - 1) * p;
            p *= r;
        }
        codes >>= 4;
    };
    middle(std::integral_constant<int, -1>{});
    mix_radix((int)(codes & 15u) + 1, [&](auto rc) __attribute__((always_inline)) {
        constexpr int R = decltype(rc)::value;
        const int nb = N / R;
        mix_stage<R, false, true, -1>(nb, nb, nb, i, NT, -1.0, tw, row, MixTurn<MUL>{row, mul});
    });
    __syncthreads();
    codes = I.codes;
    p = (int)(codes & 15u) + 1;
    tw = I.tw;
    middle(std::integral_constant<int, 1>{});
    mix_radix((int)(codes & 15u) + 1, [&](auto rc) __attribute__((always_inline)) {
        constexpr int R = decltype(rc)::value;
        const int nb = N / R;
        mix_stage<R, false, ST_LDS, 1>(nb, nb, p, i, NT, 1.0, tw, row, st);
    });
    if constexpr (ST_LDS) __syncthreads();
}

}  // namespace ifft
