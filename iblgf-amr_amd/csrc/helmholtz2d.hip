// Screened 2-D lattice Green's functions, one per spanwise Fourier mode, and
// their free-space convolution over a uniform 2-D patch of cells.
//
// For screening c > 0 (c = k dx, k the mode's spanwise wavenumber) the
// lattice Green's function of (-Lap_h + c^2) is
//   G(n, m) = 1/pi * int_0^pi cos(m x) K(x)^-n / sqrt(a^2 - 4) dx,
//   a = 4 + c^2 - 2 cos x,  K = (a + sqrt(a^2 - 4)) / 2,  n >= m >= 0,
// and the reference's kernel value is -G (lgf/helmholtz.hpp:143-153 with
// lgf/helmholtz_lookup.hpp:60-68, 146-156, 170-181: the trapezoid integral of
// (1 - cos(m x) K^-n) / (K - 1/K) minus the origin value, whose first term is
// G(0, 0)).  Both terms are evaluated here as the one integral above.
#include "capi_common.hpp"

#include <hip/hip_runtime.h>

#include <cmath>

namespace iblgf_amd {
namespace {

constexpr int    kHelmMaxModes = 256;      // modes per call (the screenings travel as a kernel argument)
constexpr long   kHelmMaxCells = 1L << 16; // nx * ny cap of the direct convolution
constexpr double kHelmMinC = 1e-4;         // smallest screening (quadrature nodes grow as 1/c)
constexpr int    kTile = 256;

struct Screenings
{
    double c[kHelmMaxModes];
};

// Trapezoid intervals on [0, pi] for screening c and lattice offsets n + m <=
// span.  The integrand is periodic and analytic in the strip |Im x| < d, d =
// acosh(1 + c^2/2) (where a^2 = 4); there |cos(m x) K^-n| <= e^{(n+m) y}, so
// the rule's error at y = d/2 is below e^{-(q - span/2) d} / c: q >= span + 45/d
// keeps it under 1e-19 relative to G(0, 0).
__host__ __device__ inline int helm_nodes(double c, int span)
{
    const double d = acosh(1.0 + 0.5 * c * c);
    const int    q = (int)ceil(span + 45.0 / d);
    return (q + 255) & ~255;
}

// table[mode][j][i] = -G_c(max(i, j), min(i, j)), 0 <= i < nx, 0 <= j < ny.
__global__ void k_helm2d_table(Screenings sc, int nmodes, int nx, int ny, double* __restrict__ table)
{
    const long per = (long)nx * ny;
    const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (t >= per * nmodes) return;
    const int    mode = (int)(t / per);
    const int    r = (int)(t - mode * per);
    const int    i = r % nx, j = r / nx;
    const int    n = i > j ? i : j, m = i > j ? j : i;
    const double c = sc.c[mode];
    const int    q = helm_nodes(c, nx + ny);
    const double h = M_PI / q;
    double       acc = 0.0;
    for (int p = 0; p <= q; ++p)
    {
        const double x = p * h;
        const double sh = sin(0.5 * x);
        const double e = c * c + 4.0 * sh * sh;  // a - 2, without cancellation near x = 0
        const double root = sqrt(e * (e + 4.0)); // sqrt(a^2 - 4)
        double       f = cos(m * x) * exp(-n * log1p(0.5 * (e + root))) / root;
        if (p == 0 || p == q) f *= 0.5;
        acc += f;
    }
    table[t] = -acc / q;
}

// dst[mode][t] = scale * sum_s table[mode][|tj - sj|][|ti - si|] * src[mode][s]
// over every cell s of the patch: one thread per target cell, the sources
// staged through LDS a tile at a time; neighbouring targets read neighbouring
// table entries.
__global__ __launch_bounds__(kTile) void k_helm2d_convolve(const double* __restrict__ table, int nx, int ny,
    const double* __restrict__ src, double* __restrict__ dst, double scale)
{
    __shared__ double s[kTile];
    const int         per = nx * ny;
    const long        off = (long)blockIdx.y * per;
    const double*     tab = table + off;
    const double*     f = src + off;
    const int         t = blockIdx.x * kTile + threadIdx.x;
    const int         ti = t % nx, tj = t / nx;
    double            acc = 0.0;
    for (int base = 0; base < per; base += kTile)
    {
        const int sidx = base + threadIdx.x;
        s[threadIdx.x] = sidx < per ? f[sidx] : 0.0;
        __syncthreads();
        if (t < per)
        {
            const int cnt = per - base < kTile ? per - base : kTile;
            int       si = base % nx, sj = base / nx;
            for (int u = 0; u < cnt; ++u)
            {
                const int dx = ti > si ? ti - si : si - ti;
                const int dy = tj > sj ? tj - sj : sj - tj;
                acc += tab[dy * nx + dx] * s[u];
                if (++si == nx)
                {
                    si = 0;
                    ++sj;
                }
            }
        }
        __syncthreads();
    }
    if (t < per) dst[off + t] = scale * acc;
}

// The same sums for patches 64 to 1024 cells wide: one workgroup per target
// row and mode, each thread up to four targets of the row; per source row the
// table row |tj - sj| and the source row are staged in LDS, so every
// multiply-add reads LDS only (the source value as a broadcast).  Sources are
// summed in index order, as above.
constexpr int kRowMin = 64, kRowMax = 4 * kTile;

__global__ __launch_bounds__(kTile) void k_helm2d_convolve_rows(const double* __restrict__ table, int nx, int ny,
    const double* __restrict__ src, double* __restrict__ dst, double scale)
{
    __shared__ double trow[kRowMax];
    __shared__ double srow[kRowMax];
    const long        off = (long)blockIdx.y * nx * ny;
    const int         tj = blockIdx.x;
    const double*     tab = table + off;
    const double*     f = src + off;
    double            acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (int sj = 0; sj < ny; ++sj)
    {
        const int dy = tj > sj ? tj - sj : sj - tj;
        for (int x = threadIdx.x; x < nx; x += kTile)
        {
            trow[x] = tab[(long)dy * nx + x];
            srow[x] = f[(long)sj * nx + x];
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            const int ti = threadIdx.x + r * kTile;
            if (ti < nx)
            {
                double a = acc[r];
                for (int si = 0; si < nx; ++si)
                {
                    const int dx = ti > si ? ti - si : si - ti;
                    a += trow[dx] * srow[si];
                }
                acc[r] = a;
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
    {
        const int ti = threadIdx.x + r * kTile;
        if (ti < nx) dst[off + (long)tj * nx + ti] = scale * acc[r];
    }
}

// The same sums for patches up to 512 cells wide with x transformed: a
// workgroup takes R target rows of a mode and walks the source rows B at a time.
// Two source rows go through one complex transform of length P >= 2 nx - 1 as real
// and imaginary part, and so do two table rows (even in x: their transforms
// are real); the transformed table rows stay in an LDS ring, because every
// step only moves the R row offsets on by B; the R target rows add up as
// spectra in registers and are transformed back at the end.  So y is summed
// directly on spectra, 2 multiply-adds a (row pair, frequency) in place of nx
// a (row pair, cell), and nothing but the patch itself is read or written: the
// call has no memory of its own.  256 x 256 cells, 8 modes: 5.50 ms by the row
// kernel above, 0.24 ms here; barriers between short transform steps bound it.
//
// The transforms are in place, radix 4 with the two radix-2 steps of each
// butterfly in natural order, so position p holds frequency k = p with its
// bits reversed.  Thread q owns position 2 q (k < P / 2; position 1 holds
// P / 2); the conjugate frequency P - k is at p with all bits below the highest
// set one flipped.
constexpr int kFftThreads = 512;

template<int LP>
struct HelmFft
{
    static constexpr int P = 1 << LP, K = P / 2;
    static constexpr int B = 4 * kFftThreads / P;       // source rows a step, one radix-4 butterfly a thread
    static constexpr int RG = kFftThreads / K;          // thread groups by target row
    static constexpr int R = RG > 8 ? RG : 8, RT = R / RG;  // target rows, of a thread
    static constexpr int need = R + B - 1;
    static constexpr int SLOTS = need <= 16 ? 16 : (need <= 32 ? 32 : 64);  // ring: row offsets alive in a step
    static_assert(SLOTS >= need && R % 2 == 0 && (R / 2 <= B || (R / 2) % B == 0), "ring and output pairs");
};

__device__ inline double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ inline double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ inline double2 cmul(double2 a, double2 w)
{
    return make_double2(fma(a.x, w.x, -a.y * w.y), fma(a.x, w.y, a.y * w.x));
}
__device__ inline double2 cmulc(double2 a, double2 w)  // a conj(w)
{
    return make_double2(fma(a.x, w.x, a.y * w.y), fma(a.y, w.x, -a.x * w.y));
}

// One transform by P / 4 threads (t) in LDS, all of the workgroup's in step.
// tw[m] = e^(-2 pi i m / P).
template<int LP, bool INVERSE>
__device__ inline void helm_fft(double2* buf, const double2* tw, int t)
{
    constexpr int P = 1 << LP, STEPS = LP / 2;
    if (INVERSE && LP % 2)
    {
#pragma unroll
        for (int h = 0; h < 2; ++h)
        {
            double2*      b = buf + 2 * (t + h * (P / 4));
            const double2 x = b[0], y = b[1];
            b[0] = cadd(x, y);
            b[1] = csub(x, y);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < STEPS; ++i)
    {
        const int     step = INVERSE ? STEPS - 1 - i : i;
        const int     len = P >> (2 * step), q = len / 4, j = t & (q - 1);
        double2*      b = buf + (t - j) * 4 + j;
        const double2 w = tw[j << (2 * step)], w2 = tw[j << (2 * step + 1)];
        const double2 a0 = b[0], a1 = b[q], a2 = b[2 * q], a3 = b[3 * q];
        if (!INVERSE)
        {
            const double2 u0 = cadd(a0, a2), u1 = cadd(a1, a3), u2 = cmul(csub(a0, a2), w);
            const double2 d = csub(a1, a3), u3 = cmul(make_double2(d.y, -d.x), w);
            b[0] = cadd(u0, u1);
            b[q] = cmul(csub(u0, u1), w2);
            b[2 * q] = cadd(u2, u3);
            b[3 * q] = cmul(csub(u2, u3), w2);
        }
        else
        {
            const double2 v1 = cmulc(a1, w2), v3 = cmulc(a3, w2);
            const double2 u0 = cadd(a0, v1), u1 = csub(a0, v1);
            const double2 u2 = cmulc(cadd(a2, v3), w), d = cmulc(csub(a2, v3), w), u3 = make_double2(-d.y, d.x);
            b[0] = cadd(u0, u2);
            b[q] = cadd(u1, u3);
            b[2 * q] = csub(u0, u2);
            b[3 * q] = csub(u1, u3);
        }
        __syncthreads();
    }
    if (!INVERSE && LP % 2)
    {
#pragma unroll
        for (int h = 0; h < 2; ++h)
        {
            double2*      b = buf + 2 * (t + h * (P / 4));
            const double2 x = b[0], y = b[1];
            b[0] = cadd(x, y);
            b[1] = csub(x, y);
        }
        __syncthreads();
    }
}

template<int LP>
__global__ __launch_bounds__(kFftThreads) void k_helm2d_convolve_fft(const double* __restrict__ table, int nx, int ny,
    const double* __restrict__ src, double* __restrict__ dst, double scale)
{
    using G = HelmFft<LP>;
    constexpr int      P = G::P, K = G::K, B = G::B, R = G::R, RT = G::RT, SLOTS = G::SLOTS;
    __shared__ double2 buf[B * P];
    __shared__ double2 tw[K];
    __shared__ double  ring[SLOTS * (K + 1)];  // [row offset mod SLOTS][q], K: frequency P / 2
    const long         off = (long)blockIdx.y * nx * ny;
    const double*      tab = table + off;
    const double*      f = src + off;
    const int          l = threadIdx.x, tj0 = blockIdx.x * R;
    const int          q = l & (K - 1), rg = l / K;          // position 2 q, target rows rg RT ..
    const int          t = l & (P / 4 - 1), mine = l / (P / 4);  // butterfly t of the step's row `mine`
    // position of the conjugate of 2 q (of position 0: P / 2, which it carries along)
    const int conj = q == 0 ? 1 : 2 * q ^ ((1 << (31 - __clz(2 * q))) - 1);
    for (int m = l; m < K; m += kFftThreads)
    {
        double sn, cs;
        sincospi(-2.0 * m / P, &sn, &cs);
        tw[m] = make_double2(cs, sn);
    }
    double2 acc[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[r] = make_double2(0.0, 0.0);
    // Transform `mine` of a step: two source rows, or the two table rows of the
    // same step (rows of one kind together: the smaller of two unlike parts would
    // take the larger's rounding).  A step's values are loaded during the step
    // before.
    const bool    is_src = mine < B / 2;
    const double* from = is_src ? f : tab;
    double        va[4], vb[4];
    auto          fetch = [&](int sj0) __attribute__((always_inline)) {
        const int     sa = sj0 + 2 * (is_src ? mine : mine - B / 2), sb = sa + 1;
        const int     ra = is_src ? sa : abs(tj0 - sa), rb = is_src ? sb : abs(tj0 - sb);
        const bool    ha = ra >= 0 && ra < ny, hb = rb >= 0 && rb < ny;
        const double *pa = from + (long)(ha ? ra : 0) * nx, *pb = from + (long)(hb ? rb : 0) * nx;
#pragma unroll
        for (int h = 0; h < 4; ++h)
        {
            const int  n = t + h * (P / 4), d = n < nx || is_src ? n : P - n;
            const bool in = d < nx;
            va[h] = in && ha ? pa[d] : 0.0;
            vb[h] = in && hb ? pb[d] : 0.0;
        }
    };
    fetch(-((R - 1 + B - 1) / B) * B);
    // the steps before row 0 only bring the ring the offsets above tj0
    for (int sj0 = -((R - 1 + B - 1) / B) * B; sj0 < ny; sj0 += B)
    {
        __syncthreads();  // the last step's spectra are no longer read
#pragma unroll
        for (int h = 0; h < 4; ++h) buf[mine * P + t + h * (P / 4)] = make_double2(va[h], vb[h]);
        fetch(sj0 + B);
        __syncthreads();
        helm_fft<LP, false>(buf + mine * P, tw, t);
        // table spectra (real each) into the ring
        for (int i = l; i < B / 2 * K; i += kFftThreads)  // i mod K is the thread's q throughout
        {
            const int     b = i / K;
            const double2 z = buf[(B / 2 + b) * P + 2 * q];
            double*       ra_ = ring + ((tj0 - (sj0 + 2 * b)) & (SLOTS - 1)) * (K + 1);
            double*       rb_ = ring + ((tj0 - (sj0 + 2 * b + 1)) & (SLOTS - 1)) * (K + 1);
            ra_[q] = z.x;
            rb_[q] = z.y;
            if (q == 0)
            {
                const double2 h = buf[(B / 2 + b) * P + 1];
                ra_[K] = h.x;
                rb_[K] = h.y;
            }
        }
        __syncthreads();
        if (sj0 < 0) continue;  // the same for the whole workgroup
#pragma unroll 1
        for (int b = 0; b < B / 2; ++b)
        {
            const double2 z = buf[b * P + 2 * q], c = buf[b * P + conj];
            // the two rows' spectra; thread 0: frequencies 0 and P / 2, both real
            double2 S[2];
            S[0] = q == 0 ? make_double2(z.x, c.x) : make_double2(0.5 * (z.x + c.x), 0.5 * (z.y - c.y));
            S[1] = q == 0 ? make_double2(z.y, c.y) : make_double2(0.5 * (z.y + c.y), 0.5 * (c.x - z.x));
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int r = 0; r < RT; ++r)
                {
                    const double* row = ring + ((tj0 + rg * RT + r - (sj0 + 2 * b + u)) & (SLOTS - 1)) * (K + 1);
                    acc[r].x = fma(row[q], S[u].x, acc[r].x);
                    acc[r].y = fma(row[q == 0 ? K : q], S[u].y, acc[r].y);
                }
        }
    }
    // two target rows a transform, as real and imaginary part
    for (int p0 = 0; p0 < R / 2; p0 += B)
    {
        __syncthreads();
#pragma unroll
        for (int odd = 0; odd < 2; ++odd)
        {
#pragma unroll
            for (int r = 0; r < RT; ++r)
            {
                const int row = rg * RT + r, b = row / 2 - p0;
                if ((row & 1) != odd || b < 0 || b >= B) continue;
                double2& z = buf[b * P + 2 * q];
                double2& c = buf[b * P + conj];
                const double2 a = acc[r];
                if (q == 0)
                {
                    if (odd) z.y = a.x, c.y = a.y;
                    else
                        z = make_double2(a.x, 0.0), c = make_double2(a.y, 0.0);
                }
                else if (odd)
                    z = make_double2(z.x - a.y, z.y + a.x), c = make_double2(c.x + a.y, c.y + a.x);
                else
                    z = a, c = make_double2(a.x, -a.y);
            }
            __syncthreads();
        }
        helm_fft<LP, true>(buf + mine * P, tw, t);
        const int row = tj0 + 2 * (p0 + mine);
        if (p0 + mine < R / 2)
            for (int n = t; n < nx; n += P / 4)
            {
                const double2 v = buf[mine * P + n];
                if (row < ny) dst[off + (long)row * nx + n] = scale / P * v.x;
                if (row + 1 < ny) dst[off + (long)(row + 1) * nx + n] = scale / P * v.y;
            }
    }
}

template<int LP>
void convolve_fft(hipStream_t s, const double* table, int nmodes, int nx, int ny, const double* src, double* dst,
    double scale)
{
    hipLaunchKernelGGL(k_helm2d_convolve_fft<LP>, dim3((unsigned)((ny + HelmFft<LP>::R - 1) / HelmFft<LP>::R), (unsigned)nmodes),
        dim3(kFftThreads), 0, s, table, nx, ny, src, dst, scale);
}

void check_shape(const char* who, int nmodes, int nx, int ny)
{
    if (nmodes < 1 || nmodes > kHelmMaxModes)
        throw std::invalid_argument(std::string(who) + ": 1 to 256 modes per call");
    if (nx < 1 || ny < 1 || (long)nx * ny > kHelmMaxCells)
        throw std::invalid_argument(std::string(who) + ": patch must hold 1 to 65536 cells");
}

void check_launch(const char* who)
{
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) throw std::runtime_error(std::string(who) + ": " + hipGetErrorString(e));
}

}  // namespace
}  // namespace iblgf_amd

using namespace iblgf_amd;
using namespace iblgf_amd::capi;

extern "C" {

int iblgf_gpu_helm2d_table(const double* c, int nmodes, int nx, int ny, double* table, void* stream)
{
    return guarded(nullptr, [&] {
        check_shape("iblgf_gpu_helm2d_table", nmodes, nx, ny);
        if (!c || !table) throw std::invalid_argument("iblgf_gpu_helm2d_table: null pointer");
        Screenings sc{};
        for (int k = 0; k < nmodes; ++k)
        {
            if (!(c[k] >= kHelmMinC) || !std::isfinite(c[k]))
                throw std::invalid_argument("iblgf_gpu_helm2d_table: screening c must be finite and >= 1e-4");
            sc.c[k] = c[k];
        }
        const long total = (long)nx * ny * nmodes;
        hipLaunchKernelGGL(k_helm2d_table, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
            (hipStream_t)stream, sc, nmodes, nx, ny, table);
        check_launch("iblgf_gpu_helm2d_table");
    });
}

int iblgf_gpu_helm2d_convolve(
    const double* table, int nmodes, int nx, int ny, const double* src, double* dst, double scale, void* stream)
{
    return guarded(nullptr, [&] {
        check_shape("iblgf_gpu_helm2d_convolve", nmodes, nx, ny);
        if (!table || !src || !dst) throw std::invalid_argument("iblgf_gpu_helm2d_convolve: null pointer");
        if (src == dst) throw std::invalid_argument("iblgf_gpu_helm2d_convolve: source and target must differ");
        const int  per = nx * ny;
        const auto st = (hipStream_t)stream;
        // Narrower, single-row and very small patches: the direct sums are faster (direct against
        // transformed, us: 4 x 4 cells, 8 modes 9.1 / 11.6; 12 x 12 9.7 / 11.0; 1 x 300 18 / 51; 2 x 2000, 2
        // modes 221 / 309; 500 x 1, 8 modes 24 / 27; 8 x 64, 4 modes 29 / 16; 16 x 16, 8 modes 16 / 11; 512 x 2
        // 45 / 27).  Wider than 512 the ring does not fit LDS.
        if (nx >= 8 && nx <= 512 && ny >= 2 && per >= 256)
        {
            if (nx <= 32) convolve_fft<6>(st, table, nmodes, nx, ny, src, dst, scale);
            else if (nx <= 64) convolve_fft<7>(st, table, nmodes, nx, ny, src, dst, scale);
            else if (nx <= 128) convolve_fft<8>(st, table, nmodes, nx, ny, src, dst, scale);
            else if (nx <= 256) convolve_fft<9>(st, table, nmodes, nx, ny, src, dst, scale);
            else
                convolve_fft<10>(st, table, nmodes, nx, ny, src, dst, scale);
        }
        else if (nx >= kRowMin && nx <= kRowMax)
            hipLaunchKernelGGL(k_helm2d_convolve_rows, dim3((unsigned)ny, (unsigned)nmodes), dim3(kTile), 0,
                (hipStream_t)stream, table, nx, ny, src, dst, scale);
        else
            hipLaunchKernelGGL(k_helm2d_convolve, dim3((unsigned)((per + kTile - 1) / kTile), (unsigned)nmodes),
                dim3(kTile), 0, (hipStream_t)stream, table, nx, ny, src, dst, scale);
        check_launch("iblgf_gpu_helm2d_convolve");
    });
}

}  // extern "C"
