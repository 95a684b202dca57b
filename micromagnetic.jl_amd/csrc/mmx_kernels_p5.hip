// mmx_kernels_p5.hip -- launchers of the last demag pass (k_p5, mmx_pass.h) for
// every transform length and epilogue variant.  Compiled once per precision
// (-DMMX_KT=double / float) so the instantiations build in parallel.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mmx_common.h"
#include "mmx_kernels.h"
#include "mmx_pass.h"

#ifndef MMX_KT
#error "compile once per precision with -DMMX_KT=double or -DMMX_KT=float"
#endif

namespace mmx {

#ifdef MMX_KT_MAIN_P5
// blocks of one last-pass launch: G.p5rx rows per block, groups rounded up to
// the 8 XCDs
int p5_grid(const DemagGeom &G)
{
    return (G.ny * ((G.nz + G.p5rx - 1) / G.p5rx) + 7) / 8 * 8;
}

// A small mesh leaves a CU two waves per SIMD or fewer in this pass, and the
// time is then the chain of dependent instructions of one wave (331x207x3 FP64:
// 1800 vector instructions in 14 us).  As long as every wave of the launch is
// resident at once (3 per SIMD), more and shorter waves are faster: 4 elements
// per thread where the rows stay wave-local, and threads beyond the rows' so
// that each takes one cell.  RK4 step, 8 elements -> 4 and more threads:
// 128x128x8 FP64 156 -> 136 us, FP32 128 -> 118; 200x50x1 Dormand-Prince 168 ->
// 151.  Launches of more waves are faster as they are (256x256x32 FP64 with
// more threads 1265 -> 1385 us; 331x207x3, whose 621 blocks of six waves do not
// all fit, 254 -> 270).  The elements per thread are the system's own (G.p5e), also
// where a batch or a band launches many copies at once: every route then rounds
// alike.  Rows and threads follow the launch.
P5Launch p5_launch(const DemagGeom &G, int copies, int e)
{
    constexpr int RESIDENT = 3 * 4 * 256;  // waves
    // (rows per block: the largest of RX, RX/2, ..., 1 that gives the launch
    // MMX_P5_MIN_BLOCKS blocks, else the one that gives the most)
    auto shape = [&](int e, P5Launch &p) {
        int rx = 1, b5 = 0;
        bool wave = false, ok = true;
#define P5S_CALL(H)                                                                                  \
    if (e == 4) {                                                                                    \
        using S = P5Shape<H, P5E4<H>::ok ? 4 : 8>;                                                   \
        rx = S::RX, b5 = S::B5, wave = S::WAVE, ok = P5E4<H>::ok;                                    \
    } else {                                                                                         \
        using S = P5Shape<H, 8>;                                                                     \
        rx = S::RX, b5 = S::B5, wave = S::WAVE;                                                      \
    }
        MMX_LG_SWITCH(G.lgH, P5S_CALL)
#undef P5S_CALL
        auto blocks = [&](int r) { return (int64_t)copies * G.ny * ((G.nz + r - 1) / r); };
        p = {e, rx, b5};
        for (int r = rx / 2; r >= 1 && blocks(p.rx) < MMX_P5_MIN_BLOCKS; r /= 2)
            if (blocks(r) > blocks(p.rx)) p.rx = r;
        const int cells = (std::min(p.rx, G.nz) * G.nx + 63) / 64 * 64;
        if (wave && cells > b5 && cells <= 512 && blocks(p.rx) * (cells / 64) <= RESIDENT) p.nt = cells;
        return ok && blocks(p.rx) * (p.nt / 64) <= RESIDENT;
    };
    P5Launch p4, p8;
    const bool small = shape(4, p4);
    shape(8, p8);
    if (!e) e = G.p5e;
    return (e ? e == 4 : small) ? p4 : p8;
}

int p5_blocks(const DemagGeom &G)
{
    DemagGeom Gl = G;
    Gl.p5rx = p5_launch(G, 1, 0).rx;
    return p5_grid(Gl);
}
#endif

template <class T>
int launch_p5(const DemagGeom &G, const cplx<T> *A, const FieldParams<T> *P, const Dyn &dyn, const Epi<T> &E,
              const T *m, int fast, uint32_t sig, const cplx<T> *tw, hipStream_t s)
{
    if (fast && sig) {
        const int gs = launch_p5_sig<T>(G, A, P, dyn, E, m, sig, tw, s);
        if (gs >= 0) return gs;
    }
    const int v = variant(E.mode, fast, E.np);
    const P5Launch p = p5_launch(G, 1, v == 5 ? 8 : 0);
    DemagGeom Gl = G;
    Gl.p5rx = p.rx;
    const int g = p5_grid(Gl);
#define P5_V(H, V, EE) hipLaunchKernelGGL((k_p5<T, H, V, 0u, false, EE>), dim3(g), dim3(p.nt), 0, s, Gl, A, P, dyn, E, m, tw)
#define P5_E(H, EE)                                                                                  \
    if (v == 4) P5_V(H, 4, EE);                                                                      \
    else if (v == 1) P5_V(H, 1, EE);                                                                 \
    else if (v == 2) P5_V(H, 2, EE);                                                                 \
    else if (v == 3) P5_V(H, 3, EE);                                                                 \
    else P5_V(H, 0, EE);
#define P5_CALL(H)                                                                                   \
    {                                                                                                \
        if (v == 5) {                                                                                \
            P5_V(H, 5, 8);                                                                           \
            break;                                                                                   \
        }                                                                                            \
        if constexpr (P5E4<H>::ok) {                                                                 \
            if (p.e == 4) {                                                                          \
                P5_E(H, 4)                                                                           \
                break;                                                                               \
            }                                                                                        \
        }                                                                                            \
        P5_E(H, 8)                                                                                   \
    }
    MMX_LG_SWITCH(G.lgH, P5_CALL)
#undef P5_CALL
#undef P5_E
#undef P5_V
    return g;
}

// Images of slot-form systems take their own kernels (V = 7: the row tile, the
// early loads and the field of the stage modes, with the cells' energies):
// 14 images of 64x64x4, FP64, 28.4 us with the term list, 11.7 in slot form.
template <class T>
void launch_p5_images(const DemagGeom &G, const cplx<T> *A, const FieldParams<T> *P, const Dyn &dyn,
                      const Epi<T> &E, const T *m, int nimg, int fast, uint32_t sig, const cplx<T> *tw,
                      hipStream_t s)
{
    const P5Launch p = p5_launch(G, nimg, 0);
    DemagGeom Gi = G;
    Gi.p5rx = p.rx;
    const dim3 g(p5_grid(Gi), nimg);
    if (fast && launch_p5_images_sig<T>(Gi, p, g, A, P, dyn, E, m, sig, tw, s)) return;
#define P5I_E(H, EE)                                                                                 \
    if (fast) hipLaunchKernelGGL((k_p5<T, H, 7, 0u, true, EE>), g, dim3(p.nt), 0, s, Gi, A, P, dyn, E, m, tw); \
    else hipLaunchKernelGGL((k_p5<T, H, 0, 0u, true, EE>), g, dim3(p.nt), 0, s, Gi, A, P, dyn, E, m, tw);
#define P5I_CALL(H)                                                                                  \
    {                                                                                                \
        if constexpr (P5E4<H>::ok) {                                                                 \
            if (p.e == 4) {                                                                          \
                P5I_E(H, 4)                                                                          \
                break;                                                                               \
            }                                                                                        \
        }                                                                                            \
        P5I_E(H, 8)                                                                                  \
    }
    MMX_LG_SWITCH(Gi.lgH, P5I_CALL)
#undef P5I_CALL
#undef P5I_E
}

template <class T>
void launch_p5_batch(const DemagGeom &G, const cplx<T> *A, int64_t astride, const int *gidx, int nmem,
                     const FieldParams<T> *const *Ps, const BatchStage<T> *st, const Dyn *dyns, int v,
                     const cplx<T> *tw, hipStream_t s)
{
    const P5Launch p = p5_launch(G, nmem, 0);
    DemagGeom Gb = G;
    Gb.p5rx = p.rx;
    const dim3 g(p5_grid(Gb), nmem), b(p.nt);
#define P5B_V(H, V, EE)                                                                              \
    hipLaunchKernelGGL((k_p5_batch<T, H, V, EE>), g, b, 0, s, Gb, A, astride, gidx, Ps, st, dyns, tw)
#define P5B_E(H, EE)                                                                                 \
    if (v == 4) P5B_V(H, 4, EE);                                                                     \
    else if (v == 1) P5B_V(H, 1, EE);                                                                \
    else if (v == 2) P5B_V(H, 2, EE);                                                                \
    else P5B_V(H, 0, EE);
#define P5B_CALL(H)                                                                                  \
    {                                                                                                \
        if constexpr (P5E4<H>::ok) {                                                                 \
            if (p.e == 4) {                                                                          \
                P5B_E(H, 4)                                                                          \
                break;                                                                               \
            }                                                                                        \
        }                                                                                            \
        P5B_E(H, 8)                                                                                  \
    }
    MMX_LG_SWITCH(Gb.lgH, P5B_CALL)
#undef P5B_CALL
#undef P5B_E
#undef P5B_V
}

template int launch_p5<MMX_KT>(const DemagGeom &, const cplx<MMX_KT> *, const FieldParams<MMX_KT> *, const Dyn &,
                               const Epi<MMX_KT> &, const MMX_KT *, int, uint32_t, const cplx<MMX_KT> *, hipStream_t);
template void launch_p5_batch<MMX_KT>(const DemagGeom &, const cplx<MMX_KT> *, int64_t, const int *, int,
                                      const FieldParams<MMX_KT> *const *, const BatchStage<MMX_KT> *, const Dyn *,
                                      int, const cplx<MMX_KT> *, hipStream_t);
template void launch_p5_images<MMX_KT>(const DemagGeom &, const cplx<MMX_KT> *, const FieldParams<MMX_KT> *,
                                       const Dyn &, const Epi<MMX_KT> &, const MMX_KT *, int, int, uint32_t,
                                       const cplx<MMX_KT> *,
                                       hipStream_t);

}  // namespace mmx
