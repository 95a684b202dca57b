// mmx_kernels_plane.hip -- the y and z transforms of the demag convolution in
// one kernel, for films of one or two layers, whose (y, z) plane of a kx column
// fits in LDS.
//
// The x-spectra of one kx column (3 components x nz rows of ny values) are
// transformed along y, convolved along z with the k-space tensor, transformed
// back along y and written to where they came from: one launch and 2 x 3 S1
// complex values of HBM traffic where the y / z / y passes take three launches
// and 2 x 3 (S1 + 2 S2).  It is bound by the latency of its one round through
// each CU (load, three exchanges per transform, store) and next by vector
// arithmetic; the 1000x1000x1 FP32 film's plane takes 46 us (its spectra, 49
// MB read and written, need 10 us at the copy rate).
#include <hip/hip_runtime.h>

#include "mmx_common.h"
#include "mmx_fft.h"
#include "mmx_kernels.h"

namespace mmx {

// Stockham stages whose values move between the threads of a sequence through
// X: fft_stage with the exchange buffer's layout and synchronisation left to
// the caller.  X.put / X.get take an element index as a thread part and a
// compile-time part that share no bits.
template <class T, int L, int E, int Ns, bool INV, class X>
__device__ __forceinline__ void fft_stages_x(cplx<T> *v, int j, const TwSet<T, L, E, Ns> &ts, const X &x)
{
    if constexpr (Ns < L) {
        constexpr int EPT = FftShape<L, E>::EPT, TPS = FftShape<L, E>::TPS;
        constexpr int Rs = TwSet<T, L, E, Ns>::Rs, NQ = EPT / Rs;
        constexpr bool LAST = Ns * Rs == L;
        cplx<T> o[LAST ? EPT : 1];
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const int jb = j + q * TPS, kk = jb & (Ns - 1);
            cplx<T> a[Rs];
#pragma unroll
            for (int r = 0; r < Rs; r++) a[r] = v[q + r * NQ];
            if constexpr (Ns > 1) {
                cplx<T> w[Rs];
                w[1] = ts.w[q];
                if (INV) w[1].y = -w[1].y;
#pragma unroll
                for (int r = 2; r < Rs; r++) w[r] = cmul(w[r >> 1], w[r - (r >> 1)]);
#pragma unroll
                for (int r = 1; r < Rs; r++) a[r] = cmul(a[r], w[r]);
            }
            dftR<T, Rs, INV>(a);
            if constexpr (LAST) {
#pragma unroll
                for (int r = 0; r < Rs; r++) o[q + r * NQ] = a[r];
            } else {
                const int base = (jb / Ns) * Ns * Rs + kk;
#pragma unroll
                for (int r = 0; r < Rs; r++) x.put(base, r * Ns, a[r]);
            }
        }
        if constexpr (LAST) {
#pragma unroll
            for (int m = 0; m < EPT; m++) v[m] = o[m];
        } else {
            x.sync();
#pragma unroll
            for (int m = 0; m < EPT; m++) v[m] = x.get(j, m * TPS);
            x.sync();
            fft_stages_x<T, L, E, Ns * Rs, INV>(v, j, ts.next, x);
        }
    }
}

// LDS a block may take: 160 KB per CU
constexpr size_t PLANE_LDS = 160 * 1024;

// Row r of the plane (one component, one z) holds element i at r*L + (swz(i) ^
// hash(r)).  LDS has 64 banks, i.e. 16 (FP64) or 32 (FP32) complex values side
// by side: the XOR with i/8 spreads the stride-8 writes of the first y stage
// over all of them and permutes aligned runs, so the accesses of the y stages
// and of the ky columns are almost free of conflicts; the row's hash does the same for
// lanes that read one ky of different z, or of different kx.  (A gap after
// every 8 elements instead makes each contiguous access wrap around the banks.
// LDS clocks per access: 6.3 at 200x50x1 FP64, 3.2 at 1000x1000x1 FP32, a twentieth
// of them conflicts; 17 with the gaps in FP64.)  swz is linear in the
// bits of i, so a compile-time part of an index costs one XOR.
template <class T, int L>
struct PlaneLds {
    static constexpr int LGB = sizeof(T) == 8 ? 4 : 5;
    static constexpr int MASK = (L < (1 << LGB) ? L : (1 << LGB)) - 1;
    static __device__ __forceinline__ constexpr int swz(int i) { return i ^ ((i >> 3) & MASK); }
};

template <class T, int L>
struct RowX {  // exchange inside a row; wave: the row's threads are lanes of one wave
    cplx<T> *pl;
    int base;       // r*L ^ hash(r)
    bool wave, on;  // on: this thread holds a sequence (the others only join the barriers)
    __device__ __forceinline__ void put(int a, int b, cplx<T> v) const
    {
        if (on) pl[(base ^ PlaneLds<T, L>::swz(a)) ^ PlaneLds<T, L>::swz(b)] = v;
    }
    __device__ __forceinline__ cplx<T> get(int a, int b) const
    {
        return pl[(base ^ PlaneLds<T, L>::swz(a)) ^ PlaneLds<T, L>::swz(b)];
    }
    __device__ __forceinline__ void sync() const
    {
        if (wave) wave_lds_sync();
        else __syncthreads();
    }
};

// z transform of length PZ = 1 or 4 over TZ neighbouring lanes, EZ elements
// each.  In: lane l holds x[l + TZ m]; out: X[m + EZ l], and the inverse takes
// it back: a transform of length EZ in the lane, the twiddle W_PZ^(l m), then a
// radix-2 butterfly across the lane pair (DPP: no LDS traffic).
template <class T, int PZ>
struct ZFft {
    static_assert(PZ == 1 || PZ == 4, "one or two layers");
    // FP64: two elements per lane keep the kernel within 128 VGPRs
    static constexpr int EZ = PZ == 1 ? 1 : (sizeof(T) == 8 ? 2 : 4), TZ = PZ / EZ;
    static constexpr int LGT = TZ - 1;
    int l;
    T sg;  // +1 in lane 0 of a pair, -1 in lane 1
    __device__ __forceinline__ explicit ZFft(int lane) : l(lane & (TZ - 1)), sg(l ? T(-1) : T(1)) {}
    __device__ __forceinline__ cplx<T> pair(cplx<T> a) const { return {quad_perm<QP_XOR1>(a.x), quad_perm<QP_XOR1>(a.y)}; }
    // W_4^(l m) of element m = 1: -i (forward) in lane 1
    template <bool INV>
    __device__ __forceinline__ cplx<T> twid(cplx<T> a) const
    {
        const cplx<T> r = mul_mi(a, INV);
        return {l ? r.x : a.x, l ? r.y : a.y};
    }
    __device__ __forceinline__ cplx<T> fly(cplx<T> a) const
    {
        const cplx<T> p = pair(a);
        return {p.x + sg * a.x, p.y + sg * a.y};
    }
    __device__ __forceinline__ void fwd(cplx<T> *v) const
    {
        dftR<T, EZ, false>(v);
        if constexpr (TZ == 2) {
            v[0] = fly(v[0]);
            v[1] = fly(twid<false>(v[1]));
        }
    }
    __device__ __forceinline__ void inv(cplx<T> *v) const
    {
        if constexpr (TZ == 2) {
            v[0] = fly(v[0]);
            v[1] = twid<true>(fly(v[1]));
        }
        dftR<T, EZ, true>(v);
    }
};

// Columns: kx = 1 .. H-1, and column 0 with kx = 0 and kx = H packed into one
// (DemagGeom::pack), so that there are H of them, a power of two like the
// chip's CUs: with H + 1 blocks of which one or two fit a CU, the last one
// cost a round of its own.
//
// Block b takes the tx consecutive kx columns from kx0 (blocks are dealt to the
// 8 XCDs round-robin; each XCD gets a contiguous run of columns, whose cache
// lines its blocks share).  Thread (s, j, t): element j of sequence s = (c, z)
// at column kx0 + t; the sequences of a column go through in batches when
// there are more of them than threads.
template <class T, int L, int PZ>
__global__ void __launch_bounds__(1024)
    k_plane(DemagGeom G, cplx<T> *__restrict__ A, const T *__restrict__ Kt, const T *__restrict__ Lline,
            const cplx<T> *__restrict__ tw, int lgtx)
{
    constexpr int EPT = FftShape<L>::EPT, TPS = FftShape<L>::TPS;
    using D = PlaneLds<T, L>;
    using Z = ZFft<T, PZ>;
    constexpr int EZ = Z::EZ, TZ = Z::TZ, TW = 64 / TZ;
    extern __shared__ __align__(16) char smem[];
    cplx<T> *pl = reinterpret_cast<cplx<T> *>(smem);
    const int nz = G.nz, ny = G.ny, KS = G.KS, Kx = G.Kx;
    const int tx = 1 << lgtx;
    const int nblk = (Kx + tx - 1) >> lgtx, per = (nblk + 7) >> 3;
    const int lb = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (lb >= nblk) return;
    const int kx0 = lb << lgtx;
    const int tid = threadIdx.x;
    const int t = tid & (tx - 1), j0 = (tid >> lgtx) & (TPS - 1), s = (tid >> lgtx) / TPS;
    const int sb = (blockDim.x >> lgtx) / TPS;  // sequences per batch
    const bool ok = kx0 + t < Kx;
    const int64_t rs = (int64_t)ny * KS;
    cplx<T> *a0 = A + (int64_t)blockIdx.y * 3 * nz * rs + kx0 + (ok ? t : 0);
    const bool wave = (TPS << lgtx) <= 64;
    const int nseq = 3 * nz;
    // LDS offset of row (t, sq) and its hash (z of neighbouring lanes, kx of
    // neighbouring threads)
    auto row_base = [&](int tt, int sq) {
        return ((tt * nseq + sq) * L) ^ (((sq & (TZ - 1)) << (D::LGB - Z::LGT)) & D::MASK) ^
               ((tt << (D::LGB - lgtx)) & D::MASK);
    };
    // ---- y forward.  In this and the loops below the thread's index passes
    // through an empty asm statement in every round: the LDS addresses and the
    // twiddle powers then belong to the round instead of being kept across all
    // of them (and the z part) in registers that the kernel does not have.
#pragma unroll 1
    for (int s0 = 0; s0 < nseq; s0 += sb) {
        int j = j0;
        asm volatile("" : "+v"(j));
        TwSet<T, L, 8> ty = fft_twiddles<T, L>(j, tw, G.lgLmax);
        const int sq = s0 + s;
        const bool act = s < sb && sq < nseq;
        const cplx<T> *src = a0 + (act ? sq : 0) * rs;
        cplx<T> v[EPT];
#pragma unroll
        for (int m = 0; m < EPT; m++) {
            const int y = j + m * TPS;
            // ny <= L/2: the upper elements are padding
            v[m] = (m < EPT / 2 && act && ok && y < ny) ? src[(int64_t)y * KS] : cplx<T>{0, 0};
        }
        const RowX<T, L> x{pl, row_base(t, act ? sq : 0), wave, act};
        ty.renew();  // (loaded with the data, not behind the exchanges)
        fft_stages_x<T, L, 8, 1, false>(v, j, ty, x);
#pragma unroll
        for (int m = 0; m < EPT; m++) x.put(j, m * TPS, v[m]);
    }
    __syncthreads();
    // ---- z: TZ lanes hold one ky column (kx0 + tt, ky); ky and its mirror
    // L - ky share the folded tensor and are taken one after the other
    {
        constexpr int Py2 = L / 2 + 1, Pz2 = PZ / 2 + 1, EL = (EZ + 1) / 2;
        const int lane = tid & 63, wv = tid >> 6, nw = blockDim.x >> 6;
        const int items = Py2 << lgtx;
        const Z zf(lane);
#pragma unroll 1
        for (int i0 = wv * TW; i0 < items; i0 += nw * TW) {
            int it = i0 + lane / TZ;
            asm volatile("" : "+v"(it));
            if (it >= items) continue;
            const int tt = it / Py2, kyf = it - tt * Py2;
            const int kx = min(kx0 + tt, Kx - 1);
            const bool two = kyf > 0 && kyf < L / 2;
            const int kym = two ? L - kyf : kyf;
            // Column 0 holds the spectra of kx = 0 and kx = H as Z = F0 + i FH.
            // Both are of real data along x, so F(-ky, z) = conj F(ky, z): the
            // first round takes F0 = (Z(ky) + conj Z(-ky))/2 with the tensor of
            // kx = 0, the second FH = (Z(ky) - conj Z(-ky))/2i with that of
            // kx = H, and the results go back to ky and -ky the same way.
            const bool packed = kx == 0;
            cplx<T> h0[3][EL];
#pragma unroll 1
            for (int half = 0; half < 2; half++) {
                if (half && !two && !packed) break;
                const int ky = half && !packed ? kym : kyf;
                const T sy = half && !packed ? T(-1) : T(1);
                cplx<T> v[3][EZ];
#pragma unroll
                for (int c = 0; c < 3; c++) {
#pragma unroll
                    for (int m = 0; m < EZ; m++) {
                        v[c][m] = cplx<T>{0, 0};
                        if (m < EL) {
                            const int z = zf.l + m * TZ, row = row_base(tt, c * nz + min(z, nz - 1));
                            cplx<T> a = pl[row ^ D::swz(ky)];
                            if (packed) {
                                const cplx<T> b = pl[row ^ D::swz(kym)];
                                a = half ? cplx<T>{T(0.5) * (a.y + b.y), T(0.5) * (b.x - a.x)}
                                         : cplx<T>{T(0.5) * (a.x + b.x), T(0.5) * (a.y - b.y)};
                            }
                            if (z < nz) v[c][m] = a;
                        }
                    }
                    zf.fwd(v[c]);
                }
                // the folded tensor: xy is odd in y, xz odd in z, yz odd in
                // both; the line tables hold what is even in them (k_convz)
                const int kt = packed && half ? G.H : kx;
                const T lxz = Lline[Pz2 + kyf], lyz = Lline[Pz2 + Py2 + kt];
                int ko = (kt * Py2 + kyf) * Pz2 * 6;
#pragma unroll
                for (int m = 0; m < EZ; m++) {
                    // (an address tied to the values before: otherwise the loads
                    // of every element start at once and hold their registers)
                    asm volatile("" : "+v"(ko), "+v"(v[2][m ? m - 1 : 0].x));
                    const int kz = m + EZ * zf.l, kzf = kz <= PZ / 2 ? kz : PZ - kz;
                    const T sz = kz <= PZ / 2 ? T(1) : T(-1);
                    const T *kb = Kt + ko + kzf * 6;
                    T k[6];
                    gld2(kb, 0, k[0], k[1]);
                    gld2(kb, 1, k[2], k[3]);
                    gld2(kb, 2, k[4], k[5]);
                    const T xx = k[0], yy = k[1], zz = k[2];
                    const T xy = sy * k[3] + Lline[kzf], xz = sz * k[4] + lxz, yz = sy * sz * k[5] + lyz;
                    const cplx<T> Mx = v[0][m], My = v[1][m], Mz = v[2][m];
                    v[0][m] = {xx * Mx.x + xy * My.x + xz * Mz.x, xx * Mx.y + xy * My.y + xz * Mz.y};
                    v[1][m] = {xy * Mx.x + yy * My.x + yz * Mz.x, xy * Mx.y + yy * My.y + yz * Mz.y};
                    v[2][m] = {xz * Mx.x + yz * My.x + zz * Mz.x, xz * Mx.y + yz * My.y + zz * Mz.y};
                }
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    zf.inv(v[c]);
#pragma unroll
                    for (int m = 0; m < EL; m++) {
                        const int z = zf.l + m * TZ;
                        if (z < nz) {
                            const int row = row_base(tt, c * nz + z);
                            const cplx<T> a = v[c][m];
                            if (!packed) {
                                pl[row ^ D::swz(ky)] = a;
                            } else if (!half) {
                                h0[c][m] = a;
                            } else {  // H0 + i HH, and conj H0 + i conj HH at -ky
                                const cplx<T> b = h0[c][m];
                                pl[row ^ D::swz(kyf)] = {b.x - a.y, b.y + a.x};
                                if (two) pl[row ^ D::swz(kym)] = {b.x + a.y, a.x - b.y};
                            }
                        }
                    }
                }
            }
        }
    }
    __syncthreads();
    // ---- y inverse
#pragma unroll 1
    for (int s0 = 0; s0 < nseq; s0 += sb) {
        int j = j0;
        asm volatile("" : "+v"(j));
        TwSet<T, L, 8> ty = fft_twiddles<T, L>(j, tw, G.lgLmax);
        const int sq = s0 + s;
        const bool act = s < sb && sq < nseq;
        const RowX<T, L> x{pl, row_base(t, act ? sq : 0), wave, act};
        cplx<T> v[EPT];
#pragma unroll
        for (int m = 0; m < EPT; m++) v[m] = x.get(j, m * TPS);
        x.sync();
        ty.renew();
        fft_stages_x<T, L, 8, 1, true>(v, j, ty, x);
        cplx<T> *dst = a0 + (act ? sq : 0) * rs;
#pragma unroll
        for (int m = 0; m < EPT / 2; m++) {
            const int y = j + m * TPS;
            if (act && ok && y < ny) dst[(int64_t)y * KS] = v[m];
        }
    }
}

// The plane kernel's launch shape for nimg systems of G; lgtx < 0: it does not
// serve G.
//
// Which meshes: one or two layers (Pz <= 4).  Measured against the three
// separate passes (us per evaluation in the passes it replaces): 1000x1000x1
// FP32 101 -> 46, 200x50x1 FP64 11.5 -> 7, 600x80x2 FP64 31.6 -> 20; with the
// z transforms of three layers and more (331x207x3, 128x128x8, FP64) it holds
// too few waves per CU and lost (50 -> 55, 25 -> 29), so those keep the passes.
//
// Columns per block: one, unless two or four still give 512 blocks (2 per CU)
// whose planes leave room for three in a CU's LDS: wider runs of kx share
// cache lines, but fewer waves cost more (1000x1000x1 FP32: two take 3 us more than one).
struct PlaneShape {
    int lgtx, threads;
    size_t lds;
};

static PlaneShape plane_shape(const DemagGeom &G, int elsize, int nimg)
{
    PlaneShape p{-1, 0, 0};
    const int L = G.Py, tps = L / 8;
    if (L < 16 || L > 2048 || G.nz > 2) return p;
    const size_t one = (size_t)3 * G.nz * L * 2 * elsize;
    if (one > PLANE_LDS) return p;
    int lg = 0;
    while (lg < 2 && (one << (lg + 1)) <= PLANE_LDS / 3 && ((int64_t)nimg * G.Kx >> (lg + 1)) >= 512) lg++;
    // sequences beyond 1024 threads go through in equal batches
    const int nseq = 3 * G.nz, batches = ((nseq * tps << lg) + 1023) / 1024;
    const int sb = (nseq + batches - 1) / batches;
    p.threads = ((sb * tps << lg) + 63) / 64 * 64;
    p.lds = one << lg;
    p.lgtx = lg;
    return p;
}

#ifdef MMX_KT_MAIN_PLANE
int plane_fits(const DemagGeom &G, int elsize) { return plane_shape(G, elsize, 1).lgtx >= 0; }
#endif

template <class T, int L, int PZ>
static void plane_call(const DemagGeom &G, const PlaneShape &p, cplx<T> *A, const T *Kt, const T *Lline, int nimg,
                       const cplx<T> *tw, hipStream_t s)
{
    const int nblk = (G.Kx + (1 << p.lgtx) - 1) >> p.lgtx;
    const dim3 grid((nblk + 7) / 8 * 8, nimg);
    if (p.lds > 65536)  // (a failure shows in the caller's check after the launch)
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&k_plane<T, L, PZ>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)PLANE_LDS);
    hipLaunchKernelGGL((k_plane<T, L, PZ>), grid, dim3(p.threads), p.lds, s, G, A, Kt, Lline, tw, p.lgtx);
}

template <class T, int L>
static void plane_z(const DemagGeom &G, const PlaneShape &p, cplx<T> *A, const T *Kt, const T *Lline, int nimg,
                    const cplx<T> *tw, hipStream_t s)
{
    // a plane of L x Pz that can never fit is not compiled
#define PLANE_Z(PZ, NZ)                                                                              \
    case PZ:                                                                                         \
        if constexpr ((size_t)3 * NZ * L * sizeof(cplx<T>) <= PLANE_LDS)                             \
            plane_call<T, L, PZ>(G, p, A, Kt, Lline, nimg, tw, s);                                   \
        break;
    switch (G.Pz) {
        PLANE_Z(1, 1)
        PLANE_Z(4, 2)
    default: break;
    }
#undef PLANE_Z
}

template <class T>
void launch_plane(const DemagGeom &G, cplx<T> *A, const T *Kt, const T *Lline, int nimg, const cplx<T> *tw,
                  hipStream_t s)
{
    const PlaneShape p = plane_shape(G, (int)sizeof(T), nimg);
    switch (G.Py) {
    case 16: plane_z<T, 16>(G, p, A, Kt, Lline, nimg, tw, s); break;
    case 32: plane_z<T, 32>(G, p, A, Kt, Lline, nimg, tw, s); break;
    case 64: plane_z<T, 64>(G, p, A, Kt, Lline, nimg, tw, s); break;
    case 128: plane_z<T, 128>(G, p, A, Kt, Lline, nimg, tw, s); break;
    case 256: plane_z<T, 256>(G, p, A, Kt, Lline, nimg, tw, s); break;
    case 512: plane_z<T, 512>(G, p, A, Kt, Lline, nimg, tw, s); break;
    case 1024: plane_z<T, 1024>(G, p, A, Kt, Lline, nimg, tw, s); break;
    case 2048: plane_z<T, 2048>(G, p, A, Kt, Lline, nimg, tw, s); break;
    default: break;
    }
}

#ifndef MMX_KT
#error "compile once per precision with -DMMX_KT=double or -DMMX_KT=float"
#endif
template void launch_plane<MMX_KT>(const DemagGeom &, cplx<MMX_KT> *, const MMX_KT *, const MMX_KT *, int,
                                   const cplx<MMX_KT> *, hipStream_t);

}  // namespace mmx
