// mmx_kernels_colr.hip -- y transforms of lengths 3 and 5 times a power of two for the separate y passes of the demag convolution.
//
// A padded length of the next power of two P carries up to 3.9 times the rows of
// a mesh of ny cells; where 5/8 P or 3/4 P hold the 2 ny - 1 rows of the
// convolution, they cut the y-z spectra, which the y and z passes move through
// memory, by as much.
#include <hip/hip_runtime.h>

#include "mmx_common.h"
#include "mmx_fft.h"
#include "mmx_kernels.h"

namespace mmx {

// kx columns per block of the length-R*M transform (M a power of two), R*M/8
// threads each: whole cache lines of kx (8 FP64, 16 FP32 values), fewer where a
// block would need more than 1024 threads
template <class T, int M, int R>
struct ColrShape {
    static constexpr int TPS = FftShape<M>::TPS, NT = R * TPS;
    static constexpr int TY0 = sizeof(T) == 8 ? 8 : 16;
    static constexpr int TY = TY0 * NT <= 1024 ? TY0 : (TY0 / 2 * NT <= 1024 ? TY0 / 2 : TY0 / 4);
    static constexpr int B = TY * NT;
    static_assert(B <= 1024, "block too large");
};

// exp(-2 pi i k/R)
template <class T, int R>
__device__ __forceinline__ constexpr cplx<T> wr(int k)
{
    constexpr double c3[2] = {-0.5, 0.86602540378443864676372317075293618};
    constexpr double c5[4] = {0.30901699437494742410229341718281906, 0.95105651629515357211643933337938214,
                              -0.80901699437494742410229341718281906, 0.58778525229247312916870595463907277};
    const double *c = R == 3 ? c3 : c5;
    k %= R;
    if (k == 0) return {T(1), T(0)};
    return 2 * k < R ? cplx<T>{(T)c[2 * k - 2], (T)-c[2 * k - 1]} : cplx<T>{(T)c[2 * (R - k) - 2], (T)c[2 * (R - k) - 1]};
}

// Length L = R*M by residues: X[R q + r] = FFT_M( W_L^(r n) sum_h W_R^(r h)
// x[n + h M] )[q].  Thread (r, j) of a column holds residue r's elements
// n = j + m TPS; X[R q + r] goes to row r*M + q (yslot).  The inverse takes the
// rows back and sums the residues' x[n + h M] in LDS.  Only n_in inputs are
// nonzero and n_out outputs wanted (convolution: half of L).
// Bound as k_coly by memory traffic at large sizes: 150x141x51 FP32 (ny = 141:
// 320 rows instead of 512) RK4 step 1056 -> 764 us.
// FULL: all L inputs are read (tensor set-up, forward only).
template <class T, int M, int R, bool INV, bool FULL = false>
__global__ void __launch_bounds__((ColrShape<T, M, R>::B)) k_colr(DemagGeom G, const cplx<T> *__restrict__ in,
                                                                 cplx<T> *__restrict__ out, int n_in, int Rin,
                                                                 int n_out, int Rout, int nplanes,
                                                                 const cplx<T> *__restrict__ tw,
                                                                 const cplx<T> *__restrict__ twl)
{
    using S = ColrShape<T, M, R>;
    constexpr int EPT = FftShape<M>::EPT, TPS = S::TPS, TY = S::TY, NT = S::NT;
    constexpr int NL = R * M / NT;  // rows per thread when the column is split over its threads
    __shared__ cplx<T> lds[TY * R * M];
    const int t = threadIdx.x % TY, q = threadIdx.x / TY, r = q / TPS, j = q % TPS;
    const int kx = blockIdx.x * TY + t;
    const int p = blockIdx.y, c = blockIdx.z;
    const int KS = G.KS;
    const bool ok = kx < G.Kx;
    const cplx<T> *src = in + ((int64_t)c * nplanes + p) * Rin * KS + (ok ? kx : 0);
    cplx<T> *dst = out + ((int64_t)c * nplanes + p) * Rout * KS + kx;
    cplx<T> v[EPT], wl[EPT];
    TwSet<T, M, 8> ts = fft_twiddles<T, M>(j, tw, G.lgLmax);
    // W_L^(r n) of this thread's elements
    auto load_wl = [&]() {
#pragma unroll
        for (int m = 0; m < EPT; m++)
            gld2(reinterpret_cast<const T *>(twl), (int64_t)r * (j + m * TPS), wl[m].x, wl[m].y);
    };
    if constexpr (!INV) {
        // the column goes to LDS once, zeros behind its n_in rows (every load and
        // every read without a branch), and each residue reads its terms there
        constexpr int NI = FULL ? NL : NL / 2, HM = FULL ? R - 1 : (R - 1) / 2;
        cplx<T> x[NI];
#pragma unroll
        for (int i = 0; i < NI; i++) x[i] = src[(int64_t)min(q + i * NT, n_in - 1) * KS];
        cplx<T> wh[HM + 1];  // W_R^(r h) = W_L^(r h M)
#pragma unroll
        for (int h = 1; h <= HM; h++)
            gld2(reinterpret_cast<const T *>(twl), (int64_t)((r * h) % R) * M, wh[h].x, wh[h].y);
        load_wl();
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const bool in = q + i * NT < n_in;
            lds[(q + i * NT) * TY + t] = cplx<T>{in ? x[i].x : T(0), in ? x[i].y : T(0)};
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < EPT; m++) {
            const int n = j + m * TPS;
            cplx<T> a = lds[n * TY + t];
#pragma unroll
            for (int h = 1; h <= HM; h++)
                // (half the column: h = (R - 1)/2 ends at n = M/2)
                if (FULL || h < HM || m < EPT / 2) a = cadd(a, cmul(lds[(n + h * M) * TY + t], wh[h]));
            v[m] = cmul(a, wl[m]);
        }
        __syncthreads();
        ts.renew();  // (loaded here, not behind the exchanges)
        fft_reg_ts<T, M, false, 8, false, TY>(v, j, lds + r * M * TY + t, ts);
        if (!ok) return;
#pragma unroll
        for (int m = 0; m < EPT; m++) {
            const int y = r * M + j + m * TPS;
            if (y < n_out) dst[(int64_t)y * KS] = v[m];
        }
    } else {
#pragma unroll
        for (int m = 0; m < EPT; m++) v[m] = src[(int64_t)(r * M + j + m * TPS) * KS];
        load_wl();
        ts.renew();
        fft_reg_ts<T, M, true, 8, false, TY>(v, j, lds + r * M * TY + t, ts);
#pragma unroll
        for (int m = 0; m < EPT; m++) {
            const cplx<T> w{wl[m].x, -wl[m].y};
            lds[(r * M + j + m * TPS) * TY + t] = cmul(v[m], w);
        }
        __syncthreads();
        if (!ok) return;
#pragma unroll
        for (int i = 0; i < NL; i++) {
            const int y = q + i * NT;
            if (i * NT >= n_out) break;
            const int h = y / M, n = y % M;
            cplx<T> a{0, 0};
#pragma unroll
            for (int hh = 0; hh < R; hh++)
                if (h == hh) {  // (a block's threads share h but at its edges)
#pragma unroll
                    for (int rr = 0; rr < R; rr++) {
                        const cplx<T> z = lds[(rr * M + n) * TY + t];
                        cplx<T> w = wr<T, R>(rr * hh);
                        w.y = -w.y;
                        a = rr * hh % R == 0 ? cadd(a, z) : cadd(a, cmul(z, w));
                    }
                }
            if (y < n_out) dst[(int64_t)y * KS] = a;
        }
    }
}

template <class T, int M, int R>
static void colr_call(const DemagGeom &G, const cplx<T> *in, cplx<T> *out, int n_in, int Rin, int n_out, int Rout,
                      int nplanes, int ncomp, int inverse, const cplx<T> *tw, hipStream_t s)
{
    using S = ColrShape<T, M, R>;
    const dim3 grid((G.Kx + S::TY - 1) / S::TY, nplanes, ncomp);
    const cplx<T> *twl = static_cast<const cplx<T> *>(G.twy);
    if (inverse)
        hipLaunchKernelGGL((k_colr<T, M, R, true>), grid, dim3(S::B), 0, s, G, in, out, n_in, Rin, n_out, Rout, nplanes,
                           tw, twl);
    else if (2 * n_in > G.Py) {
        if constexpr (sizeof(T) == 8)  // the set-up runs in FP64
            hipLaunchKernelGGL((k_colr<T, M, R, false, true>), grid, dim3(S::B), 0, s, G, in, out, n_in, Rin, n_out,
                               Rout, nplanes, tw, twl);
    } else
        hipLaunchKernelGGL((k_colr<T, M, R, false>), grid, dim3(S::B), 0, s, G, in, out, n_in, Rin, n_out, Rout,
                           nplanes, tw, twl);
}

template <class T, int R>
static void colr_m(const DemagGeom &G, const cplx<T> *in, cplx<T> *out, int n_in, int Rin, int n_out, int Rout,
                   int nplanes, int ncomp, int inverse, const cplx<T> *tw, hipStream_t s)
{
#define COLR_M(M)                                                                                    \
    case M: colr_call<T, M, R>(G, in, out, n_in, Rin, n_out, Rout, nplanes, ncomp, inverse, tw, s); break;
    switch (G.Py / R) {
        COLR_M(16)
        COLR_M(32)
        COLR_M(64)
        COLR_M(128)
        COLR_M(256)
    default: break;
    }
#undef COLR_M
}

template <class T>
void launch_colr(const DemagGeom &G, const cplx<T> *in, cplx<T> *out, int n_in, int Rin, int n_out, int Rout,
                 int nplanes, int ncomp, int inverse, const cplx<T> *tw, hipStream_t s)
{
    if (G.Ry == 3) colr_m<T, 3>(G, in, out, n_in, Rin, n_out, Rout, nplanes, ncomp, inverse, tw, s);
    else if (G.Ry == 5) colr_m<T, 5>(G, in, out, n_in, Rin, n_out, Rout, nplanes, ncomp, inverse, tw, s);
}

#ifndef MMX_KT
#error "compile once per precision with -DMMX_KT=double or -DMMX_KT=float"
#endif
template void launch_colr<MMX_KT>(const DemagGeom &, const cplx<MMX_KT> *, cplx<MMX_KT> *, int, int, int, int, int, int,
                                  int, const cplx<MMX_KT> *, hipStream_t);

}  // namespace mmx
