// dcm_spectral.hip -- the inverse of the pressure operator by fast
// transforms, as the preconditioner of the mixed path's FP32 inner solve
// (dcm_set_precond_multigrid on grids uniform along every axis).
//
// On such a grid, which is every grid the reference makes
// (initialisation.f90:429-446), the operator of mat_ax (dynamics.f90:187-229,
// periodic in x and y, the Neumann copy in z) is a sum of three second
// differences with constant coefficients.  A discrete Hartley transform along
// x and along y (real, its own inverse; the second difference is a symmetric
// circulant) and a cosine transform (DCT-II) along z diagonalise it, so
//     M t = C^-1 H H diag(1/lambda) H H C t,   lambda(0,0,0) -> 0,
// is its inverse on vectors of zero mean, a fixed linear map as BiCGSTAB
// requires.  With FP32 rounding the inner solve then needs one iteration
// where the V-cycle needs two to six; the FP64 refinement around it decides
// convergence, as with every preconditioner.
//
// Five launches, each reading and writing the vector once: DCT along k with
// the right-hand side formed on the way in, Hartley along j, Hartley - scale
// - Hartley along i, Hartley along j, inverse DCT with p = x + bet*p on the
// way out.  A block holds a tile of whole lines, [position][column], in LDS;
// two neighbouring real lines form one complex line, and a complex FFT of
// mixed radix (8, 4, 2, 3, 5, 7) runs in place, decimation in frequency,
// leaving the spectrum in digit-reversed order, from which the Hartley (or cosine) coefficients of
// the two lines are read; the scaled spectrum goes back by decimation in
// time.  Bound by the strided lines' memory traffic above a million cells
// (512x512x256, beside the advection: 270 to 430 us a pass of 0.54 GB) and by
// the passes' latency below (128x96x64: 7 to 10 us each).
// Measured, a mixed solve to 1e-10 with the V-cycle and with this: 128x96x64
// 1594 -> 456 us, 112x112x80 1664 -> 649, 64x160x128 1792 -> 530; a model step
// at 256x256x128 (9 tracers) 6.00 -> 4.14 ms, at 512x512x256 34.5 -> 23.7.
#include <cmath>
#include <algorithm>
#include <vector>

#include "dcm_device.h"

namespace dcm {

namespace {

constexpr int kMaxStages = 10;
constexpr int kMaxLine = 1024;  // a tile of 8 lines and its tables: 50 KiB of LDS
constexpr int kSpThreads = 256;

// the transform of one axis
struct Axis {
    int n, ns;
    int radix[kMaxStages];
    unsigned magic[kMaxStages];  // floor(u / M) = umulhi(u, magic), M the sub-line
    const float2 *tw;            // exp(-2 pi i t / n)
    const unsigned short *rev;   // position of coefficient m after the DIF stages
};
struct SpTab {
    Axis x, y, z;
    const float *lx, *ly, *lz;   // eigenvalues along each axis
    const float2 *cs;            // (cos, sin)(pi l / (2 kp))
    float norm;
    unsigned kmagic;             // floor(2 e / kp) = umulhi(e, kmagic)
};

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
    return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ float2 cadd(float2 a, float2 b) {
    return make_float2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ float2 csub(float2 a, float2 b) {
    return make_float2(a.x - b.x, a.y - b.y);
}
__device__ __forceinline__ float2 mi(float2 a) { return make_float2(a.y, -a.x); }  // -i a

// the DFT of R values in natural order
template <int R> struct Dft {
    static __device__ __forceinline__ void run(float2 (&a)[R], const float2 *tw, int n) {
        float2 o[R];
        const int st = n / R;
#pragma unroll
        for (int q = 0; q < R; ++q) {
            float2 s = a[0];
#pragma unroll
            for (int p = 1; p < R; ++p) s = cadd(s, cmul(a[p], tw[((p * q) % R) * st]));
            o[q] = s;
        }
#pragma unroll
        for (int q = 0; q < R; ++q) a[q] = o[q];
    }
};
template <> struct Dft<2> {
    static __device__ __forceinline__ void run(float2 (&a)[2], const float2 *, int) {
        const float2 t = a[1];
        a[1] = csub(a[0], t);
        a[0] = cadd(a[0], t);
    }
};
template <> struct Dft<4> {
    static __device__ __forceinline__ void run(float2 (&a)[4], const float2 *, int) {
        const float2 s02 = cadd(a[0], a[2]), d02 = csub(a[0], a[2]);
        const float2 s13 = cadd(a[1], a[3]), d13 = mi(csub(a[1], a[3]));
        a[0] = cadd(s02, s13);
        a[1] = cadd(d02, d13);
        a[2] = csub(s02, s13);
        a[3] = csub(d02, d13);
    }
};
template <> struct Dft<8> {
    static __device__ __forceinline__ void run(float2 (&a)[8], const float2 *, int) {
        float2 e[4] = {a[0], a[2], a[4], a[6]}, o[4] = {a[1], a[3], a[5], a[7]};
        Dft<4>::run(e, nullptr, 0);
        Dft<4>::run(o, nullptr, 0);
        const float h = 0.70710678118654752f;
        o[1] = make_float2(h * (o[1].x + o[1].y), h * (o[1].y - o[1].x));
        o[2] = mi(o[2]);
        o[3] = make_float2(h * (o[3].y - o[3].x), -h * (o[3].x + o[3].y));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            a[q] = cadd(e[q], o[q]);
            a[q + 4] = csub(e[q], o[q]);
        }
    }
};

// One stage over every complex column of the tile z[pos][1 << lcp], positions
// ld apart: blocks of L = R*M positions.  DIF: DFT then twiddles; DIT:
// twiddles then DFT.
template <int R, bool DIT>
__device__ __forceinline__ void stage(float2 *z, const float2 *tw, int n, int M, unsigned magic,
                                      int lcp, int ld) {
    const int items = (n / R) << lcp, st = n / (R * M);
    for (int it = threadIdx.x; it < items; it += kSpThreads) {
        const int c = it & ((1 << lcp) - 1), u = it >> lcp;
        const int b = M == 1 ? u : (int)__umulhi((unsigned)u, magic), t = u - b * M;
        float2 *p = z + (b * R * M + t) * ld + c;
        float2 a[R];
#pragma unroll
        for (int q = 0; q < R; ++q) {
            a[q] = p[q * M * ld];
            if (DIT && q > 0) a[q] = cmul(a[q], tw[t * q * st]);
        }
        Dft<R>::run(a, tw, n);
#pragma unroll
        for (int q = 0; q < R; ++q) {
            if (!DIT && q > 0) a[q] = cmul(a[q], tw[t * q * st]);
            p[q * M * ld] = a[q];
        }
    }
    __syncthreads();
}
template <bool DIT>
__device__ __forceinline__ void run_stage(float2 *z, const float2 *tw, const Axis &A, int s, int M, int lcp, int ld) {
    const unsigned mg = A.magic[s];
    switch (A.radix[s]) {
        case 2: stage<2, DIT>(z, tw, A.n, M, mg, lcp, ld); break;
        case 3: stage<3, DIT>(z, tw, A.n, M, mg, lcp, ld); break;
        case 4: stage<4, DIT>(z, tw, A.n, M, mg, lcp, ld); break;
        case 5: stage<5, DIT>(z, tw, A.n, M, mg, lcp, ld); break;
        case 7: stage<7, DIT>(z, tw, A.n, M, mg, lcp, ld); break;
        default: stage<8, DIT>(z, tw, A.n, M, mg, lcp, ld); break;
    }
}
// natural order -> digit-reversed
__device__ __forceinline__ void fft_dif(float2 *z, const float2 *tw, const Axis &A, int lcp, int ld) {
    int L = A.n;
    for (int s = 0; s < A.ns; ++s) {
        L /= A.radix[s];
        run_stage<false>(z, tw, A, s, L, lcp, ld);
    }
}
// digit-reversed -> natural order
__device__ __forceinline__ void fft_dit(float2 *z, const float2 *tw, const Axis &A, int lcp, int ld) {
    int M = 1;
    for (int s = A.ns - 1; s >= 0; --s) {
        run_stage<true>(z, tw, A, s, M, lcp, ld);
        M *= A.radix[s];
    }
}

// Hartley coefficient m of the first (x) and second (y) line of a complex
// column from the spectrum's values at m and n-m
__device__ __forceinline__ float2 hartley(float2 zm, float2 zn) {
    return make_float2(0.5f * ((zm.x + zn.x) + (zn.y - zm.y)),
                       0.5f * ((zm.y + zn.y) + (zm.x - zn.x)));
}

// the line of pair e of a run of lines along z
__device__ __forceinline__ int line_of(const SpTab &T, int e) {
    return T.z.n == 2 ? e : (int)__umulhi((unsigned)e, T.kmagic);
}

__device__ __forceinline__ bool stopped(const SolverScalars *sc) {
    return sc->breakdown != 0 || sc->done != 0;
}

// Consecutive blocks go to the eight XCDs in turn; a tile narrower than a
// 128-byte line shares its lines with its neighbours, which therefore run on
// the same XCD: each takes a run of tiles
__device__ __forceinline__ int tile_id() {
    const int nb = gridDim.x, b = blockIdx.x;
    return (nb & 7) == 0 ? (b & 7) * (nb >> 3) + (b >> 3) : b;
}

// A block's LDS: the tile z, then the axis's twiddles and positions, which
// every stage and both ends of a transform look up
struct Tile {
    float2 *z;
    const float2 *tw;
    const unsigned short *rev;
};
__device__ __forceinline__ Tile tile_of(unsigned char *lds, const Axis &A, int cells) {
    float2 *z = (float2 *)lds, *tw = z + cells;
    unsigned short *rev = (unsigned short *)(tw + A.n);
    for (int t = threadIdx.x; t < A.n; t += kSpThreads) {
        tw[t] = A.tw[t];
        rev[t] = A.rev[t];
    }
    return {z, tw, rev};
}

// Hartley transform along y, in place: columns (i, k), lines of jp values kp
// apart; two neighbours along k (kp is even) are a complex column.  cp = 1 <<
// lcp: complex columns of the tile.
__global__ __launch_bounds__(kSpThreads) void k_sp_y(float *v, SpTab T, int ip, int kp, int lcp,
                                                     const SolverScalars *sc) {
    extern __shared__ __align__(16) unsigned char sp_lds[];
    if (stopped(sc)) return;
    const Axis &A = T.y;
    const int n = A.n, cp = 1 << lcp, q = threadIdx.x & (cp - 1);
    const Tile L = tile_of(sp_lds, A, n << lcp);
    const int kh = kp / 2, col = tile_id() * cp + q;
    const bool act = col < ip * kh;
    const int i = act ? col / kh : 0;
    float2 *g = (float2 *)v + (size_t)i * n * kh + (act ? col - i * kh : 0);
    const int p0 = threadIdx.x >> lcp, ps = kSpThreads >> lcp;
#pragma unroll 8
    for (int p = p0; p < n; p += ps)
        L.z[(p << lcp) + q] = act ? g[(size_t)p * kh] : make_float2(0.f, 0.f);
    __syncthreads();
    fft_dif(L.z, L.tw, A, lcp, cp);
#pragma unroll 4
    for (int m = p0; m < n; m += ps) {
        const float2 h = hartley(L.z[(L.rev[m] << lcp) + q], L.z[(L.rev[m ? n - m : 0] << lcp) + q]);
        if (act) g[(size_t)m * kh] = h;
    }
}

// Hartley along x, division by the eigenvalues, Hartley back, in place:
// columns (j, k) of ip values jp*kp apart
__global__ __launch_bounds__(kSpThreads) void k_sp_x(float *v, SpTab T, int jp, int kp, int lcp,
                                                     const SolverScalars *sc) {
    extern __shared__ __align__(16) unsigned char sp_lds[];
    if (stopped(sc)) return;
    const Axis &A = T.x;
    const int n = A.n, cp = 1 << lcp, q = threadIdx.x & (cp - 1);
    const Tile L = tile_of(sp_lds, A, n << lcp);
    const int kh = kp / 2, col = tile_id() * cp + q, ncol = jp * kh;
    const bool act = col < ncol;
    float2 *g = (float2 *)v + (act ? col : 0);
    const int p0 = threadIdx.x >> lcp, ps = kSpThreads >> lcp;
#pragma unroll 8
    for (int p = p0; p < n; p += ps)
        L.z[(p << lcp) + q] = act ? g[(size_t)p * ncol] : make_float2(0.f, 0.f);
    const int j = act ? col / kh : 0, k = act ? 2 * (col - j * kh) : 0;
    const float l0 = T.ly[j] + T.lz[k], l1 = T.ly[j] + T.lz[k + 1];
    __syncthreads();
    fft_dif(L.z, L.tw, A, lcp, cp);
    // scale coefficients m and n-m of both lines, in their digit-reversed
    // places
    for (int m = p0; m <= n / 2; m += ps) {
        const float s0 = T.lx[m] + l0, s1 = T.lx[m] + l1;
        const float w0 = s0 != 0.f ? T.norm / s0 : 0.f, w1 = s1 != 0.f ? T.norm / s1 : 0.f;
        float2 *a = L.z + (L.rev[m] << lcp) + q, *b = L.z + (L.rev[m ? n - m : 0] << lcp) + q;
        const float2 za = *a, zb = *b;
        const float2 ha = hartley(za, zb), hb = hartley(zb, za);
        *a = make_float2(w0 * ha.x, w1 * ha.y);
        *b = make_float2(w0 * hb.x, w1 * hb.y);
    }
    __syncthreads();
    fft_dit(L.z, L.tw, A, lcp, cp);
#pragma unroll 4
    for (int p = p0; p < n; p += ps) {
        const float2 h = hartley(L.z[(p << lcp) + q], L.z[((p ? n - p : 0) << lcp) + q]);
        if (act) g[(size_t)p * ncol] = h;
    }
}

// The right-hand side t = r - bet*(omg*v1) (MODE 0, dynamics.f90:394) or s =
// r - alf*v1 (MODE 1, :405, stored to t_out) and its DCT-II along z into v.
// Columns are the ip*jp lines of kp consecutive values; level 2h of a line
// is position h of its FFT, level 2h+1 position n-1-h.  The tile's positions
// are one complex value further apart than its columns, against bank
// conflicts of the transposed access.
template <int MODE>
__global__ __launch_bounds__(kSpThreads) void k_sp_z_fwd(const float *__restrict__ r,
                                                         const float *__restrict__ v1,
                                                         float *__restrict__ t_out,
                                                         float *__restrict__ v, SpTab T,
                                                         int ncol, int lcp,
                                                         const SolverScalars *sc) {
    extern __shared__ __align__(16) unsigned char sp_lds[];
    if (stopped(sc)) return;
    const Axis &A = T.z;
    const int n = A.n, nh = n / 2, ct = 2 << lcp, ld = (1 << lcp) + 1;
    const Tile L = tile_of(sp_lds, A, n * ld);
    float *f = (float *)L.z;
    const float a = MODE == 0 ? (float)sc->bet : (float)sc->alf, bo = (float)sc->omg;
    const bool vz = MODE == 0 && sc->iters == 0;  // v1 = 0 (dynamics.f90:380)
    const int c0 = blockIdx.x * ct, nc = min(ct, ncol - c0);
    // lines are consecutive in memory: a tile is one run of nc*n values
    const size_t base = (size_t)c0 * nh;
    const float2 *r2 = (const float2 *)r + base, *v2 = (const float2 *)v1 + base;
#pragma unroll 4
    for (int e = threadIdx.x; e < ct * nh; e += kSpThreads) {
        const int c = line_of(T, e), h = e - c * nh;
        float2 t = make_float2(0.f, 0.f);
        if (c < nc) {
            const float2 rv = r2[e], vv = vz ? t : v2[e];
            t = MODE == 0 ? make_float2(rv.x - a * (bo * vv.x), rv.y - a * (bo * vv.y))
                          : make_float2(rv.x - a * vv.x, rv.y - a * vv.y);
            if (MODE == 1) ((float2 *)t_out + base)[e] = t;
        }
        f[2 * h * ld + c] = t.x;
        f[2 * (n - 1 - h) * ld + c] = t.y;
    }
    __syncthreads();
    fft_dif(L.z, L.tw, A, lcp, ld);
    auto coef = [&](int l, int c) {
        const float2 zm = L.z[L.rev[l] * ld + (c >> 1)], zn = L.z[L.rev[l ? n - l : 0] * ld + (c >> 1)];
        const float re = (c & 1) ? 0.5f * (zm.y + zn.y) : 0.5f * (zm.x + zn.x);
        const float im = (c & 1) ? 0.5f * (zn.x - zm.x) : 0.5f * (zm.y - zn.y);
        const float2 cs = T.cs[l];
        return re * cs.x + im * cs.y;
    };
#pragma unroll 2
    for (int e = threadIdx.x; e < nc * nh; e += kSpThreads) {
        const int c = line_of(T, e), h = e - c * nh;
        ((float2 *)v + base)[e] = make_float2(coef(2 * h, c), coef(2 * h + 1, c));
    }
}

// The inverse DCT of v along z into out (P: out = x + bet*out, the search
// direction's update, dynamics.f90:399)
template <bool P>
__global__ __launch_bounds__(kSpThreads) void k_sp_z_inv(const float *__restrict__ v,
                                                         float *__restrict__ out, SpTab T,
                                                         int ncol, int lcp,
                                                         const SolverScalars *sc) {
    extern __shared__ __align__(16) unsigned char sp_lds[];
    if (stopped(sc)) return;
    const Axis &A = T.z;
    const int n = A.n, nh = n / 2, ct = 2 << lcp, ld = (1 << lcp) + 1;
    const Tile L = tile_of(sp_lds, A, n * ld);
    const float *f = (const float *)L.z;
    const float bet = P ? (float)sc->bet : 0.f;
    const bool pread = P && sc->iters != 0;  // p = 0 (dynamics.f90:379)
    const int c0 = blockIdx.x * ct, nc = min(ct, ncol - c0);
    const size_t base = (size_t)c0 * n;
    // the conjugate of exp(i pi l/(2 n)) [(Ca_l + Cb_{n-l}) + i (Cb_l -
    // Ca_{n-l})], C_n = 0, for l and n-l at once (l = h of 0..n/2-1, and the
    // thread of h = 0 also takes n/2)
    auto put = [&](int l, float x, float y) {
        const float2 cs = T.cs[l];
        return make_float2(x * cs.x - y * cs.y, -(x * cs.y + y * cs.x));
    };
#pragma unroll 2
    for (int e = threadIdx.x; e < nh << lcp; e += kSpThreads) {
        const int q = line_of(T, e), l = e - q * nh, ln = l ? n - l : nh;
        const bool act = 2 * q < nc, act2 = 2 * q + 1 < nc;
        const float *va = v + base + (size_t)(2 * q) * n, *vb = va + n;
        const float al = act ? va[l] : 0.f, an = act ? va[ln] : 0.f;
        const float bl = act2 ? vb[l] : 0.f, bn = act2 ? vb[ln] : 0.f;
        L.z[l * ld + q] = l ? put(l, al + bn, bl - an) : put(0, al, bl);
        L.z[ln * ld + q] = l ? put(ln, an + bl, bn - al) : put(nh, an + bn, bn - an);
    }
    __syncthreads();
    fft_dif(L.z, L.tw, A, lcp, ld);
    float2 *o = (float2 *)(out + base);
#pragma unroll 4
    for (int e = threadIdx.x; e < nc * nh; e += kSpThreads) {
        const int c = line_of(T, e), h = e - c * nh;
        const float s = (c & 1) ? -1.f : 1.f;
        float2 x = make_float2(s * f[2 * L.rev[h] * ld + c], s * f[2 * L.rev[n - 1 - h] * ld + c]);
        if (P) {
            const float2 p = pread ? o[e] : make_float2(0.f, 0.f);
            x = make_float2(x.x + bet * p.x, x.y + bet * p.y);
        }
        o[e] = x;
    }
}

// radices of n, largest first; false when a factor above 7 remains
bool factor(int n, std::vector<int> &f) {
    f.clear();
    for (int r : {8, 4, 2, 7, 5, 3})
        while (n % r == 0 && n > 1) {
            // 16 is 4 x 4, not 8 x 2
            const int q = r == 8 && n == 16 ? 4 : r;
            f.push_back(q);
            n /= q;
        }
    return n == 1 && f.size() <= (size_t)kMaxStages;
}

}  // namespace

struct Spectral {
    SpTab T{};
    void *mem = nullptr;
    // along x, y, z: log2 of a tile's complex columns, tiles, LDS bytes
    int lcp[3] = {};
    unsigned tiles[3] = {};
    size_t lds[3] = {};
};

void sp_release(dcm_ctx *c) {
    Spectral *S = (Spectral *)c->sp;
    if (!S) return;
    (void)hipFree(S->mem);
    delete S;
    c->sp = nullptr;
}

// The transforms' tables, when the grid allows them: constant spacings along
// every axis, line lengths of at most 1024 with factors 2, 3, 5 and 7 only
// (a larger factor would make its stage a direct sum of as many terms).
// The caller leaves grids with a thin axis to the V-cycle -- a semi-coarsened
// hierarchy, or one that ends at one cell along some axis -- although this is
// faster there too (a 512x4x256 step 3.6 ms against 0.6): the two agree in p
// up to its undetermined constant, which these transforms keep and the
// V-cycle's rounding lets wander, on such grids by up to 1.2e-6 of p in one
// solve and 4e-6 within the first steps, more than the 3e-7 (a solve) and 2e-6
// (a step) within which the choice of the preconditioner may move p.  Over 80
// grids of the others it was 2e-8 at the median and 3e-7 at most.  (That is
// not the mixed path's distance from the FP64 path, which FP32 advection
// sets: at 256x256x128 p is 2e-8 off after two steps and 2.4e-6 after 27,
// the same with either preconditioner and with the Chebyshev sweeps.)
int sp_prepare(dcm_ctx *c) {
    if (c->sp) return DCM_OK;
    const Geo &g = c->geo;
    auto constant = [](const std::vector<double> &a) {
        for (double x : a)
            if (x != a[0]) return false;
        return true;
    };
    for (const std::vector<double> *a :
         {&c->h_dx, &c->h_dxn, &c->h_dy, &c->h_dyn, &c->h_dz, &c->h_dzn})
        if (!constant(*a)) return DCM_OK;
    const int n[3] = {g.ip, g.jp, g.kp};
    std::vector<int> f[3];
    for (int a = 0; a < 3; ++a)
        if (n[a] > kMaxLine || !factor(n[a], f[a])) return DCM_OK;
    if ((long long)n[0] * n[1] * n[2] >= (1LL << 31)) return DCM_OK;
    // one table: twiddles, DCT factors, eigenvalues (FP64, rounded once), rev
    std::vector<float> h;
    size_t tw[3], lam[3], cs, rev[3];
    const double coef[3] = {1.0 / (c->h_dx[0] * c->h_dxn[0]), 1.0 / (c->h_dy[0] * c->h_dyn[0]),
                            1.0 / (c->h_dz[0] * c->h_dzn[0])};
    const double pi = 3.14159265358979323846;
    for (int a = 0; a < 3; ++a) {
        tw[a] = h.size();
        for (int t = 0; t < n[a]; ++t) {
            h.push_back((float)std::cos(2.0 * pi * t / n[a]));
            h.push_back((float)-std::sin(2.0 * pi * t / n[a]));
        }
    }
    cs = h.size();
    for (int l = 0; l < n[2]; ++l) {
        h.push_back((float)std::cos(pi * l / (2.0 * n[2])));
        h.push_back((float)std::sin(pi * l / (2.0 * n[2])));
    }
    for (int a = 0; a < 3; ++a) {
        lam[a] = h.size();
        for (int m = 0; m < n[a]; ++m) {
            // -4 sin^2(pi m / n), along z -4 sin^2(pi m / (2 n))
            const double s = std::sin(pi * m / (a == 2 ? 2.0 * n[a] : (double)n[a]));
            h.push_back((float)(-4.0 * s * s * coef[a]));
        }
    }
    Spectral *S = new Spectral();
    Axis *ax[3] = {&S->T.x, &S->T.y, &S->T.z};
    for (int a = 0; a < 3; ++a) {
        rev[a] = h.size();
        std::vector<unsigned short> r(2 * ((n[a] + 1) / 2));
        for (int m = 0; m < n[a]; ++m) {
            // after the stages f[0], f[1], ... the first digit of m (base
            // f[0]) is the most significant of the position
            int q = m, L = n[a], p = 0;
            for (int d : f[a]) {
                L /= d;
                p += (q % d) * L;
                q /= d;
            }
            r[m] = (unsigned short)p;
        }
        const size_t o = h.size();
        h.resize(o + r.size() / 2);
        std::copy((const char *)r.data(), (const char *)(r.data() + r.size()), (char *)&h[o]);
        Axis &A = *ax[a];
        A.n = n[a];
        A.ns = (int)f[a].size();
        int L = n[a];
        for (int s = 0; s < A.ns; ++s) {
            A.radix[s] = f[a][s];
            L /= f[a][s];
            // exact for u < 2^16 and M >= 2: u * (2^32/M + 1) / 2^32
            A.magic[s] = L > 1 ? (unsigned)((1ULL << 32) / L + 1) : 0u;
        }
        // lines per tile, a power of two: up to 8192 values, a quarter of a
        // CU's LDS, so that four blocks hide each other's loads and barriers
        // (at 512x512x256 k_sp_y 277 us and k_sp_x 427, with 64 KiB tiles of
        // whole 128-byte lines 546 and 1454, both beside the advection);
        // fewer on a grid of less than 512 tiles
        const long long cols = (long long)n[0] * n[1] * n[2] / n[a];
        int ct = 8;
        while (ct < 256 && ct * 2 * n[a] <= 8192) ct *= 2;
        while (ct > 8 && (cols + ct - 1) / ct < 512) ct /= 2;
        while ((2 << S->lcp[a]) < ct) ++S->lcp[a];
        S->tiles[a] = (unsigned)((cols + ct - 1) / ct);
        S->lds[a] = ((size_t)n[a] * (ct / 2 + (a == 2)) + n[a]) * sizeof(float2) +
                    n[a] * sizeof(unsigned short);
    }
    if (hipMalloc(&S->mem, h.size() * sizeof(float)) != hipSuccess) {
        delete S;
        set_error("spectral preconditioner: out of device memory");
        return DCM_OUT_OF_MEMORY;
    }
    c->sp = S;
    float *d = (float *)S->mem;
    if (hipMemcpy(d, h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) {
        sp_release(c);
        return DCM_HIP_ERROR;
    }
    for (int a = 0; a < 3; ++a) {
        ax[a]->tw = (const float2 *)(d + tw[a]);
        ax[a]->rev = (const unsigned short *)(d + rev[a]);
    }
    S->T.cs = (const float2 *)(d + cs);
    S->T.lx = d + lam[0];
    S->T.ly = d + lam[1];
    S->T.lz = d + lam[2];
    // Hartley twice: 1/n each; the inverse DCT as an FFT: 1/kp
    S->T.kmagic = n[2] > 2 ? (unsigned)((1ULL << 32) / (n[2] / 2) + 1) : 0u;
    S->T.norm = (float)(1.0 / ((double)n[0] * n[1] * n[2]));
    return DCM_OK;
}

// out = M t (mode 1: t = r - alf*v1, stored to t_out) or out = M t + bet*out
// (mode 0: t = r - bet*(omg*v1)); v: scratch.
int sp_apply(dcm_ctx *c, int mode, const float *r, const float *v1, float *t_out, float *v,
             float *out, const SolverScalars *sc) {
    Spectral *S = (Spectral *)c->sp;
    const Geo &g = c->geo;
    const int lines = g.ip * g.jp;
    auto grid = [&](int a) { return dim3(S->tiles[a]); };
    const dim3 block(kSpThreads);
    const int tok = prof_begin(c, "spectral");
    if (mode == 0)
        hipLaunchKernelGGL(k_sp_z_fwd<0>, grid(2), block, S->lds[2], c->stream, r, v1, t_out, v,
                           S->T, lines, S->lcp[2], sc);
    else
        hipLaunchKernelGGL(k_sp_z_fwd<1>, grid(2), block, S->lds[2], c->stream, r, v1, t_out, v,
                           S->T, lines, S->lcp[2], sc);
    hipLaunchKernelGGL(k_sp_y, grid(1), block, S->lds[1], c->stream, v, S->T, g.ip, g.kp,
                       S->lcp[1], sc);
    hipLaunchKernelGGL(k_sp_x, grid(0), block, S->lds[0], c->stream, v, S->T, g.jp, g.kp,
                       S->lcp[0], sc);
    hipLaunchKernelGGL(k_sp_y, grid(1), block, S->lds[1], c->stream, v, S->T, g.ip, g.kp,
                       S->lcp[1], sc);
    if (mode == 0)
        hipLaunchKernelGGL(k_sp_z_inv<true>, grid(2), block, S->lds[2], c->stream,
                           (const float *)v, out, S->T, lines, S->lcp[2], sc);
    else
        hipLaunchKernelGGL(k_sp_z_inv<false>, grid(2), block, S->lds[2], c->stream,
                           (const float *)v, out, S->T, lines, S->lcp[2], sc);
    DCM_LAUNCH_CHECK();
    prof_end(c, tok);
    return DCM_OK;
}

}  // namespace dcm
