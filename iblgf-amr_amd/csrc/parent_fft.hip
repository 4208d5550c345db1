// Far and near field of one level by transforms of whole parents.
//
// In an FMM pass of the Laplace kernel every level-L target block sums over
// all level-L source blocks among the children of its parent's 27
// neighbours (Fmm::compute_influence_field, include/iblgf/fmm/fmm.hpp:988-1027:
// near neighbours and influence list together), sources taken without their
// boundary ring.  So the eight children of a parent are one source of
// (2e)^3 points and, with one ring, one target of (2e + 2)^3 points, and the
// level is a sum over parent pairs: 27 spectral products of a parent in place
// of 8 x 216 of blocks.  A transform of length P >= 4e + 1 keeps the cyclic
// images out of the target.  On a 4290-block adaptive tree of 16^3 cells the
// level-L work of a solve takes 2.5 ms (FP64, one stream); transforms and
// products of blocks took 6.1 ms.
//
// A leg of length P = R1 R2, R1 and R2 without common factor, is a prime-factor
// transform: with n = R2 a + R1 b (mod P) and k1 = k mod R1, k2 = k mod R2,
//   X[k1, k2] = sum_b w2^(b k2) sum_a w1^(a k1) x[n]
// has no twiddle factors between its two steps.  One thread computes one line
// for one k1 (forward) or one a (inverse): the step of length R1 straight from
// the inputs that are not zero, then the step of length R2 in registers with
// its inputs folded, x_b + x_{R2-b} and x_b - x_{R2-b}, which halves its
// products.  x and y frequencies are stored in the order q = k2 R1 + k1, so
// that the threads of a wave always store next to each other.
#include "kernels.hpp"

#include <algorithm>
#include <stdexcept>

namespace iblgf_amd {
namespace {

// P is the smallest length above 4e with two such factors and R2 odd (e = 6:
// 26, 8: 33, 10: 42, 14: 57, 16: 65); a spectrum grows with its cube.
template<int N> struct Factors;
template<> struct Factors<8> { static constexpr int R1 = 2, R2 = 13; };
template<> struct Factors<10> { static constexpr int R1 = 3, R2 = 11; };
template<> struct Factors<12> { static constexpr int R1 = 6, R2 = 7; };
template<> struct Factors<16> { static constexpr int R1 = 3, R2 = 19; };
template<> struct Factors<18> { static constexpr int R1 = 5, R2 = 13; };

template<int N>
struct Par
{
    static constexpr int n = N, E = N - 2;
    static constexpr int M = 2 * E;  // source points a side
    static constexpr int W = M + 2;  // target points a side
    static constexpr int R1 = Factors<N>::R1, R2 = Factors<N>::R2;
    static constexpr int P = R1 * R2, H = P / 2 + 1;
    static constexpr int PP = P * P, NF = H * PP;
    static constexpr int NCH = (NF + 63) / 64;  // chunks of 64 frequencies
    static constexpr int NN = N * N, N3 = N * N * N;
    // A plane's workgroup: one thread per (line, k1) of the longer leg.
    static constexpr int T = (P * R1 + 63) / 64 * 64;
    // Odd row lengths in LDS: 16-byte stores one row apart meet different banks.
    static constexpr int PS = P | 1, WS = W | 1;
    static_assert(P >= M + W - 1 && R2 % 2 == 1, "transform length");
};

// ---------------------------------------------------------------------------
// Roots of unity as constants: cos and sin of 2 pi j / r from their Taylor
// sums after reduction to an eighth of the circle by exact fractions.
// ---------------------------------------------------------------------------
struct CosSin
{
    double c, s;
};
constexpr CosSin cos_sin_small(double x, double lo)
{
    const double y = x * x;
    double       c = 1.0, s = 1.0;
    for (int k = 13; k >= 1; --k)
    {
        c = 1.0 - y / ((2 * k - 1) * (2 * k)) * c;
        s = 1.0 - y / ((2 * k) * (2 * k + 1)) * s;
    }
    s *= x;
    return {c - lo * s, s + lo * c};
}
constexpr CosSin root(int j, int r)
{
    j %= r;
    int  num = j, den = r;
    bool ns = false, nc = false, sw = false;
    if (2 * num > den)
    {
        num = den - num;
        ns = true;
    }
    if (4 * num > den)  // pi - x
    {
        num = den - 2 * num;
        den = 2 * den;
        nc = true;
    }
    if (8 * num > den)  // pi / 2 - x
    {
        num = den - 4 * num;
        den = 4 * den;
        sw = true;
    }
    const double   q = (double)num / den;
    const CosSin   v = cos_sin_small(6.283185307179586 * q, 2.4492935982947064e-16 * q);
    const double   c = sw ? v.s : v.c, s = sw ? v.c : v.s;
    return {nc ? -c : c, ns ? -s : s};
}
template<int R>
struct Roots
{
    double c[R] = {}, s[R] = {};
    constexpr Roots()
    {
        for (int j = 0; j < R; ++j)
        {
            const CosSin v = root(j, R);
            c[j] = v.c;
            s[j] = v.s;
        }
    }
};
template<int R>
inline constexpr Roots<R> kRoots{};

// k[k1][k2]: the frequency with k mod R1 = k1 and k mod R2 = k2.
template<int R1, int R2>
struct Crt
{
    int k[R1][R2] = {};
    constexpr Crt()
    {
        for (int f = 0; f < R1 * R2; ++f) k[f % R1][f % R2] = f;
    }
};
template<int R1, int R2>
inline constexpr Crt<R1, R2> kCrt{};

// v -> out(k, X_k), X_k = sum_b v_b e^(SIGN 2 pi i b k / R), R odd.
template<int R, int SIGN, class Out>
__device__ inline void small_dft(double2 (&v)[R], Out&& out)
{
    constexpr int h = (R - 1) / 2;
    double2       x0 = v[0];
#pragma unroll
    for (int j = 1; j <= h; ++j)
    {
        const double2 a = v[j], b = v[R - j];
        v[j] = make_double2(a.x + b.x, a.y + b.y);
        v[R - j] = make_double2(a.x - b.x, a.y - b.y);
        x0.x += v[j].x;
        x0.y += v[j].y;
    }
    out(0, x0);
#pragma unroll
    for (int k = 1; k <= h; ++k)
    {
        double2 C = v[0], D = make_double2(0.0, 0.0);
#pragma unroll
        for (int j = 1; j <= h; ++j)
        {
            constexpr int r = R;
            const double  c = kRoots<r>.c[(j * k) % r], s = kRoots<r>.s[(j * k) % r];
            C.x = fma(c, v[j].x, C.x);
            C.y = fma(c, v[j].y, C.y);
            D.x = fma(s, v[r - j].x, D.x);
            D.y = fma(s, v[r - j].y, D.y);
        }
        if (SIGN > 0)
        {
            out(k, make_double2(C.x - D.y, C.y + D.x));
            out(R - k, make_double2(C.x + D.y, C.y - D.x));
        }
        else
        {
            out(k, make_double2(C.x + D.y, C.y - D.x));
            out(R - k, make_double2(C.x - D.y, C.y + D.x));
        }
    }
}

// w[a] = e^(SIGN 2 pi i a k / R) for the thread's k.
template<int R, int SIGN>
__device__ inline void leg_roots(int k, const double2* tab, double2 (&w)[R])
{
#pragma unroll
    for (int a = 1; a < R; ++a)
    {
        w[a] = tab[(a * k) % R];
        if (SIGN < 0) w[a].y = -w[a].y;
    }
}

__device__ inline void cfma(double2 a, double2 w, double2& s)
{
    s.x = fma(a.x, w.x, fma(-a.y, w.y, s.x));
    s.y = fma(a.x, w.y, fma(a.y, w.x, s.y));
}

// First step of a forward leg: v_b = sum_a w1^(a k1) x[n], inputs n < M only.
template<int N, class Load>
__device__ inline void forward_first(const double2 (&w)[Par<N>::R1], double2 (&v)[Par<N>::R2], Load&& load)
{
    using G = Par<N>;
#pragma unroll
    for (int b = 0; b < G::R2; ++b)
    {
        double2 s = make_double2(0.0, 0.0);
#pragma unroll
        for (int a = 0; a < G::R1; ++a)
        {
            const int n = (G::R2 * a + G::R1 * b) % G::P;
            if (n >= G::M) continue;
            const double2 x = load(n);
            if (a == 0)
            {
                s.x += x.x;
                s.y += x.y;
            }
            else if (G::R1 == 2)
            {
                s.x = fma(w[a].x, x.x, s.x);
                s.y = fma(w[a].x, x.y, s.y);
            }
            else
                cfma(x, w[a], s);
        }
        v[b] = s;
    }
}

// The step of length R1 of an inverse leg, in place: v_a = sum_{k1} w1^(-a k1) v_{k1}.
template<int R>
__device__ inline void inverse_first(double2 (&v)[R])
{
    if constexpr (R == 2)
    {
        const double2 a = v[0], b = v[1];
        v[0] = make_double2(a.x + b.x, a.y + b.y);
        v[1] = make_double2(a.x - b.x, a.y - b.y);
    }
    else if constexpr (R == 6)
    {
        double2 e[3] = {v[0], v[2], v[4]}, o[3] = {v[1], v[3], v[5]}, E[3], O[3];
        small_dft<3, 1>(e, [&](int k, double2 X) { E[k] = X; });
        small_dft<3, 1>(o, [&](int k, double2 X) { O[k] = X; });
#pragma unroll
        for (int k = 0; k < 3; ++k)
        {
            double2 t = make_double2(0.0, 0.0);
            cfma(O[k], make_double2(kRoots<6>.c[k], kRoots<6>.s[k]), t);
            v[k] = make_double2(E[k].x + t.x, E[k].y + t.y);
            v[k + 3] = make_double2(E[k].x - t.x, E[k].y - t.y);
        }
    }
    else
    {
        double2 u[R];
        small_dft<R, 1>(v, [&](int k, double2 X) { u[k] = X; });
#pragma unroll
        for (int k = 0; k < R; ++k) v[k] = u[k];
    }
}

template<int R>
__device__ inline void root_table(double2* tab)
{
    if (threadIdx.x == 0)
    {
#pragma unroll
        for (int j = 0; j < R; ++j) tab[j] = make_double2(kRoots<R>.c[j], kRoots<R>.s[j]);
    }
}

template<class T> struct Spec;
template<> struct Spec<double>
{
    using C = double2;
    static __device__ inline double2 get(double2 v) { return v; }
    static __device__ inline double2 put(double2 v) { return v; }
};
template<> struct Spec<float>
{
    using C = float2;
    static __device__ inline double2 get(float2 v) { return make_double2(v.x, v.y); }
    static __device__ inline float2  put(double2 v) { return make_float2((float)v.x, (float)v.y); }
};

constexpr int kLineThreads = 256;

// Spectra are stored by chunks of 64 frequencies, in a chunk by parent: the
// products read a chunk's sources from one stretch of memory.  (Parent by
// parent, their rows of 1 KB lay 2 MB apart at n = 18: twice the time.)
// chunk0: the first chunk that is stored.
__device__ inline size_t spec_at(int f, int chunk0, int row, int rows)
{
    return ((size_t)((f >> 6) - chunk0) * rows + row) * 64 + (f & 63);
}

// The kz planes [z0, z0 + nz) of one round of a pass and the chunks they lie
// in.  Frequencies are independent of each other between the z legs, so a
// pass whose spectra do not fit its scratch takes them some planes at a time;
// an outer chunk's other planes are neither written nor read.
//
// The storage type of a plane (T double: FP64 for all): with T float, planes
// below zl are FP64 and the others FP32, the FP32 chunks behind the FP64
// ones; a chunk that holds planes of both is stored as both.
struct Slice
{
    int z0, nz, zl;
    int chunk0, nchunk;    // of the planes [z0, zl)
    int chunk0f, nchunkf;  // of the planes [zl, z0 + nz)
};
// The FP32 chunks of a spectrum array.
__device__ inline const float2* low_part(const double2* spec, const Slice& sl, int rows)
{
    return reinterpret_cast<const float2*>(spec + (size_t)sl.nchunk * rows * 64);
}
__device__ inline float2* low_part(double2* spec, const Slice& sl, int rows)
{
    return reinterpret_cast<float2*>(spec + (size_t)sl.nchunk * rows * 64);
}

// ---------------------------------------------------------------------------
// Forward z leg (real to half spectrum): mid[item][kz][y][x], item = component
// * count + parent.  One thread per column of a parent, the whole transform in
// its registers; its points come from the two children below and above (an
// absent child is zero).  Real input: k1 and R1 - k1 give conjugate
// frequencies, so only k1 <= R1 / 2 is computed.  Memory bounds it: 0.65 GB in
// 0.13 ms a 4290-block solve (a dense matrix from scalar registers: 0.32 ms).
// PART: only planes [z0, z0 + nz) are kept; otherwise all H of them.
// ---------------------------------------------------------------------------
template<int N, bool PART>
__global__ __launch_bounds__(kLineThreads) void k_parent_fwd_z(const double* __restrict__ src, long fcs,
    const int* __restrict__ child, int count, int ncomp, double2* __restrict__ mid, int z0, int nz)
{
    using G = Par<N>;
    constexpr int E = G::E, M = G::M, MM = M * M, R1 = G::R1, R2 = G::R2, P = G::P, h = (R2 - 1) / 2;
    const long    q = (long)blockIdx.x * kLineThreads + threadIdx.x;
    const int     item = (int)(q / MM), col = (int)(q - (long)item * MM);
    if (item >= count * ncomp) return;
    const int c = item / count, p = item - c * count;
    const int y = col / M, x = col - y * M, cy = y / E, cx = x / E;
    const int lo = child[8 * p + cx + 2 * cy], hi = child[8 * p + cx + 2 * cy + 4];
    src += c * fcs + G::NN + (y - cy * E + 1) * N + (x - cx * E + 1);
    double in[M];
#pragma unroll
    for (int a = 0; a < E; ++a) in[a] = lo >= 0 ? src[(size_t)lo * G::N3 + a * G::NN] : 0.0;
#pragma unroll
    for (int a = 0; a < E; ++a) in[E + a] = hi >= 0 ? src[(size_t)hi * G::N3 + a * G::NN] : 0.0;
    double2*   out = mid + (size_t)item * (PART ? nz : G::H) * MM + col;
    const auto put = [&](int k, double2 X) {
        if (!PART) out[(size_t)k * MM] = X;
        else if (k >= z0 && k < z0 + nz)
            out[(size_t)(k - z0) * MM] = X;
    };
#pragma unroll
    for (int k1 = 0; 2 * k1 <= R1; ++k1)
    {
        if (k1 == 0 || 2 * k1 == R1)  // real sums
        {
            double u[R2];
#pragma unroll
            for (int b = 0; b < R2; ++b)
            {
                u[b] = 0.0;
#pragma unroll
                for (int a = 0; a < R1; ++a)
                {
                    const int n = (R2 * a + R1 * b) % P;
                    if (n < M) u[b] += (k1 * a) % 2 ? -in[n] : in[n];
                }
            }
            double s0 = u[0];
#pragma unroll
            for (int j = 1; j <= h; ++j)
            {
                const double t = u[j] + u[R2 - j], d = u[j] - u[R2 - j];
                u[j] = t;
                u[R2 - j] = d;
                s0 += t;
            }
            put(kCrt<R1, R2>.k[k1][0], make_double2(s0, 0.0));
#pragma unroll
            for (int k2 = 1; k2 <= h; ++k2)
            {
                double C = u[0], D = 0.0;
#pragma unroll
                for (int j = 1; j <= h; ++j)
                {
                    C = fma(kRoots<R2>.c[(j * k2) % R2], u[j], C);
                    D = fma(kRoots<R2>.s[(j * k2) % R2], u[R2 - j], D);
                }
                const int k = kCrt<R1, R2>.k[k1][k2];
                if (k < G::H) put(k, make_double2(C, -D));
                else
                    put(P - k, make_double2(C, D));
            }
        }
        else
        {
            double2 v[R2];
#pragma unroll
            for (int b = 0; b < R2; ++b)
            {
                v[b] = make_double2(0.0, 0.0);
#pragma unroll
                for (int a = 0; a < R1; ++a)
                {
                    const int n = (R2 * a + R1 * b) % P;
                    if (n >= M) continue;
                    v[b].x = a == 0 ? v[b].x + in[n] : fma(kRoots<R1>.c[(a * k1) % R1], in[n], v[b].x);
                    if (a > 0) v[b].y = fma(-kRoots<R1>.s[(a * k1) % R1], in[n], v[b].y);
                }
            }
            small_dft<R2, -1>(v, [&](int k2, double2 X) {
                const int k = kCrt<R1, R2>.k[k1][k2];
                if (k < G::H) put(k, X);
                else
                    put(P - k, make_double2(X.x, -X.y));
            });
        }
    }
}

// ---------------------------------------------------------------------------
// Forward y and x legs of one (parent, component, kz) plane: spectrum
// frequency (kz, qx, qy).  Writes of the spectra bound it: 2.1 GB at 3.6 TB/s
// (0.59 ms) for the 954 source parents of a 4290-block solve of 16^3 cells in
// FP64.  Five waves a SIMD let three workgroups share a CU at n = 18.
// ---------------------------------------------------------------------------
template<int N, class T>
__global__ __launch_bounds__(Par<N>::T) __attribute__((amdgpu_waves_per_eu(5))) void k_parent_fwd_plane(
    const double2* __restrict__ mid, double2* __restrict__ spec, int rows, Slice sl)
{
    using G = Par<N>;
    constexpr int      M = G::M, P = G::P, R1 = G::R1, R2 = G::R2, PS = G::PS;
    __shared__ double2 in[M * M];   // [y][x]
    __shared__ double2 Y[M * PS];   // [x][qy]
    __shared__ double2 tab[R1];
    const int          l = threadIdx.x, zl = blockIdx.x / rows, row = blockIdx.x - zl * rows, kz = sl.z0 + zl;
    mid += ((size_t)row * sl.nz + zl) * (M * M);
    root_table<R1>(tab);
    for (int q = l; q < M * M; q += G::T) in[q] = mid[q];
    __syncthreads();
    double2 w[R1], v[R2];
    if (l < M * R1)
    {
        const int k1 = l / M, x = l - k1 * M;
        leg_roots<R1, -1>(k1, tab, w);
        forward_first<N>(w, v, [&](int n) { return in[n * M + x]; });
        small_dft<R2, -1>(v, [&](int k2, double2 X) { Y[x * PS + k2 * R1 + k1] = X; });
    }
    __syncthreads();
    if (l < P * R1)
    {
        const int k1 = l / P, qy = l - k1 * P;
        leg_roots<R1, -1>(k1, tab, w);
        forward_first<N>(w, v, [&](int n) { return Y[n * PS + qy]; });
        const int f = kz * G::PP + k1 * P + qy;
        if (sizeof(T) == 8 || kz < sl.zl)  // the same for the whole workgroup
            small_dft<R2, -1>(
                v, [&](int k2, double2 X) { spec[spec_at(f + k2 * (R1 * P), sl.chunk0, row, rows)] = X; });
        else
        {
            float2* out = low_part(spec, sl, rows);
            small_dft<R2, -1>(v, [&](int k2, double2 X) {
                out[spec_at(f + k2 * (R1 * P), sl.chunk0f, row, rows)] = Spec<float>::put(X);
            });
        }
    }
}

// ---------------------------------------------------------------------------
// Spectral products: tspec[target] = sum over its entries of
// ghat[offset] * sspec[source].  A workgroup takes 64 frequencies and a run of
// (target group, component) pairs, a wave one pair at a time; the 27 kernel
// values of a frequency are in LDS (the 13 with a leading negative offset are
// the conjugates of their opposites: the point kernel is even), and a row of
// zeros for the targets of a group that a source does not reach.  Products and
// sums are FP64 for either storage type.  The workgroups that share a chunk
// of frequencies are neighbours on one XCD: a source's line is read from
// memory once, and by its other groups from that L2.  Four targets share a
// load of a source (2.2 targets on average in a 4290-block tree; 1.8 products
// are issued for each that counts); skipping the others by a branch each put
// an LDS wait into every branch.  One target a wave: 1.19 ms a solve of 4290
// blocks in FP64, 2.28 for three components in FP32; four: 1.06 and 1.83
// (branches: 1.07 and 2.04).  The spectra read and written once are 0.54 and
// 0.80 ms of that at the rate of a copy.
// ---------------------------------------------------------------------------
constexpr int kMacWaves = 8;

template<int U, class T>
__device__ inline void mac_entries(const int2* __restrict__ ent, int& e, int end,
    const typename Spec<T>::C* __restrict__ sp, const double2* Gs, double2 (&acc)[4])
{
    for (; e + U <= end; e += U)
    {
        int2                id[U];
        typename Spec<T>::C S[U];
#pragma unroll
        for (int i = 0; i < U; ++i) id[i] = ent[e + i];
#pragma unroll
        for (int i = 0; i < U; ++i) S[i] = sp[(size_t)id[i].x * 64];
#pragma unroll
        for (int i = 0; i < U; ++i)
#pragma unroll
            for (int t = 0; t < 4; ++t) cfma(Spec<T>::get(S[i]), Gs[((id[i].y >> 8 * t) & 255) * 64], acc[t]);
    }
}

// The products of one chunk: T is its storage type.
template<class T>
__device__ inline void mac_chunk(const int4* __restrict__ group, const int* __restrict__ begin,
    const int2* __restrict__ ent, int ngroup, int ntgt, int nsrc, int ncomp, const double2* Gs,
    const typename Spec<T>::C* __restrict__ sspec, typename Spec<T>::C* __restrict__ tspec, int chunk, int seg, int nseg)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int npair = ngroup * ncomp, per = (npair + nseg - 1) / nseg, lo = seg * per, hi = min(lo + per, npair);
    for (int pr = lo + wave; pr < hi; pr += kMacWaves)
    {
        const int  c = pr / ngroup, g = pr - c * ngroup;
        const int  end = begin[g + 1];
        int        e = begin[g];
        const int4 to = group[g];
        const typename Spec<T>::C* sp = sspec + ((size_t)chunk * ncomp + c) * nsrc * 64 + lane;
        typename Spec<T>::C*       tp = tspec + ((size_t)chunk * ncomp + c) * ntgt * 64 + lane;
        double2 acc[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = make_double2(0.0, 0.0);
        mac_entries<8, T>(ent, e, end, sp, Gs + lane, acc);
        mac_entries<2, T>(ent, e, end, sp, Gs + lane, acc);
        mac_entries<1, T>(ent, e, end, sp, Gs + lane, acc);
        if (to.x >= 0) tp[(size_t)to.x * 64] = Spec<T>::put(acc[0]);
        if (to.y >= 0) tp[(size_t)to.y * 64] = Spec<T>::put(acc[1]);
        if (to.z >= 0) tp[(size_t)to.z * 64] = Spec<T>::put(acc[2]);
        if (to.w >= 0) tp[(size_t)to.w * 64] = Spec<T>::put(acc[3]);
    }
}

template<class T>
__global__ __launch_bounds__(64 * kMacWaves) void k_parent_mac(const int4* __restrict__ group,
    const int* __restrict__ begin, const int2* __restrict__ ent, int ngroup, int ntgt, int nsrc, int ncomp, const double2* __restrict__ ghat,
    const double2* __restrict__ sspec, double2* __restrict__ tspec, Slice sl, int nseg)
{
    __shared__ double2 Gs[(kParentNone + 1) * 64];
    const int          r = blockIdx.x >> 3, chunk = (r / nseg) * 8 + (blockIdx.x & 7), seg = r % nseg;
    if (chunk >= sl.nchunk + sl.nchunkf) return;  // the whole workgroup
    const bool fine = sizeof(T) == 8 || chunk < sl.nchunk;
    const int  lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int  gc = fine ? sl.chunk0 + chunk : sl.chunk0f + chunk - sl.nchunk;  // chunk of the whole spectrum
    if (wave == kMacWaves - 1) Gs[kParentNone * 64 + lane] = make_double2(0.0, 0.0);
    for (int o = wave; o < 27; o += kMacWaves)
    {
        // stored: offsets 13 (own parent) to 26; offset o < 13 is the opposite of 26 - o
        double2 g = ghat[((size_t)gc * 14 + (o < 13 ? 13 - o : o - 13)) * 64 + lane];
        if (o < 13) g.y = -g.y;
        Gs[o * 64 + lane] = g;
    }
    __syncthreads();
    if (fine) mac_chunk<double>(group, begin, ent, ngroup, ntgt, nsrc, ncomp, Gs, sspec, tspec, chunk, seg, nseg);
    else
        mac_chunk<float>(group, begin, ent, ngroup, ntgt, nsrc, ncomp, Gs, low_part(sspec, sl, nsrc * ncomp),
            low_part(tspec, sl, ntgt * ncomp), chunk - sl.nchunk, seg, nseg);
}

// ---------------------------------------------------------------------------
// Inverse x and y legs of one (parent, component, kz) plane, restricted to the
// target's window: mid[item][kz][y][x], y and x < W (window point i is
// point i - 1 of the parent).  All inputs count here, so a leg is two rounds:
// the step of length R1 in place (the x leg's straight from memory, each value
// read once), then the step of length R2.  The x leg's outputs wait in
// registers while its inputs are still read: both share one LDS buffer.  A
// round over all inputs per output residue, as forward, reads LDS five times
// as often and took 0.53 ms where this takes 0.37 (n = 18, 451 targets, FP64).
// ---------------------------------------------------------------------------
template<int N>
__device__ inline int window(int a, int b)  // window point of (a, b), W or more: outside
{
    using G = Par<N>;
    int n = G::R2 * a + G::R1 * b;
    if (n >= G::P) n -= G::P;
    return n == G::P - 1 ? 0 : n + 1;
}

template<int N, class T>
__global__ __launch_bounds__(Par<N>::T) void k_parent_inv_plane(
    const double2* __restrict__ spec, double2* __restrict__ mid, int rows, Slice sl)
{
    using G = Par<N>;
    constexpr int      P = G::P, R1 = G::R1, R2 = G::R2, W = G::W, WS = G::WS;
    static_assert(P * WS <= G::PP, "the x leg's outputs take the place of its inputs");
    __shared__ double2 buf[G::PP];  // [k2][a][qy], then [qy][x]
    const int          l = threadIdx.x, zl = blockIdx.x / rows, row = blockIdx.x - zl * rows, kz = sl.z0 + zl;
    mid += ((size_t)row * G::H + kz) * (W * W);
    double2 u[R1], v[R2];
    const auto first = [&](auto load) {
        for (int it = l; it < R2 * P; it += G::T)
        {
            const int k2 = it / P, at = k2 * (R1 * P) + it - k2 * P;
#pragma unroll
            for (int k = 0; k < R1; ++k) u[k] = load(kz * G::PP + at + k * P);
            inverse_first<R1>(u);
#pragma unroll
            for (int k = 0; k < R1; ++k) buf[at + k * P] = u[k];
        }
    };
    if (sizeof(T) == 8 || kz < sl.zl)  // the same for the whole workgroup
        first([&](int f) { return spec[spec_at(f, sl.chunk0, row, rows)]; });
    else
    {
        const float2* in = low_part(spec, sl, rows);
        first([&](int f) { return Spec<float>::get(in[spec_at(f, sl.chunk0f, row, rows)]); });
    }
    __syncthreads();
    const int a = l / P, qy = l - a * P;
    if (l < P * R1)
    {
#pragma unroll
        for (int k = 0; k < R2; ++k) v[k] = buf[k * (R1 * P) + l];
    }
    __syncthreads();
    if (l < P * R1)
        small_dft<R2, 1>(v, [&](int b, double2 X) {
            const int i = window<N>(a, b);
            if (i < W) buf[qy * WS + i] = X;
        });
    __syncthreads();
    for (int it = l; it < R2 * W; it += G::T)
    {
        const int k2 = it / W, at = k2 * (R1 * WS) + it - k2 * W;
#pragma unroll
        for (int k = 0; k < R1; ++k) u[k] = buf[at + k * WS];
        inverse_first<R1>(u);
#pragma unroll
        for (int k = 0; k < R1; ++k) buf[at + k * WS] = u[k];
    }
    __syncthreads();
    if (l < W * R1)
    {
        const int ay = l / W, x = l - ay * W;
#pragma unroll
        for (int k = 0; k < R2; ++k) v[k] = buf[(k * R1 + ay) * WS + x];
        small_dft<R2, 1>(v, [&](int b, double2 X) {
            const int i = window<N>(ay, b);
            if (i < W) mid[i * W + x] = X;
        });
    }
}

// ---------------------------------------------------------------------------
// Inverse z leg (half spectrum to real), added into the children: one thread
// per column of a child pair (below and above), which holds the column's
// frequencies and the whole column of the window; points of two children's
// rings are computed by each.  0.63 GB in 0.15 ms a 4290-block solve (a dense
// matrix: 0.43 ms).
// ---------------------------------------------------------------------------
template<int N>
__global__ __launch_bounds__(kLineThreads) void k_parent_inv_z(const double2* __restrict__ mid,
    const int* __restrict__ child, int count, int ncomp, double* __restrict__ dst, long fcs, double scale)
{
    using G = Par<N>;
    constexpr int E = G::E, W = G::W, WW = W * W, R1 = G::R1, R2 = G::R2, P = G::P, H = G::H, h = (R2 - 1) / 2;
    const long    q = (long)blockIdx.x * kLineThreads + threadIdx.x;
    const int     item = (int)(q / (4 * G::NN)), r = (int)(q - (long)item * (4 * G::NN));
    if (item >= count * ncomp) return;
    const int c = item / count, p = item - c * count;
    const int cxy = r / G::NN, ji = r - cxy * G::NN, j = ji / N, i = ji - j * N;
    const int lo = child[8 * p + cxy], hi = child[8 * p + cxy + 4];
    if (lo < 0 && hi < 0) return;
    const double2* in = mid + (size_t)item * H * WW + ((cxy >> 1) * E + j) * W + (cxy & 1) * E + i;
    double2        X[H];
#pragma unroll
    for (int k = 0; k < H; ++k) X[k] = in[(size_t)k * WW];
    double acc[W];
#pragma unroll
    for (int a = 0; a < R1; ++a)
    {
        // y_{k2} = sum_{k1} w1^(-a k1) X[k1, k2]; the outputs are real, so y_{R2 - k2} is its conjugate
        double  y0 = 0.0;
        double2 y[h + 1];
#pragma unroll
        for (int k2 = 0; k2 <= h; ++k2)
        {
            double2 s = make_double2(0.0, 0.0);
#pragma unroll
            for (int k1 = 0; k1 < R1; ++k1)
            {
                const int     k = kCrt<R1, R2>.k[k1][k2];
                const double2 x = k < H ? X[k < H ? k : 0] : make_double2(X[k < H ? 0 : P - k].x, -X[k < H ? 0 : P - k].y);
                const double  cw = kRoots<R1>.c[(a * k1) % R1], sw = kRoots<R1>.s[(a * k1) % R1];
                if ((a * k1) % R1 == 0)
                {
                    s.x += x.x;
                    if (k2 > 0) s.y += x.y;
                }
                else
                {
                    s.x = fma(cw, x.x, fma(-sw, x.y, s.x));
                    if (k2 > 0) s.y = fma(sw, x.x, fma(cw, x.y, s.y));
                }
            }
            if (k2 == 0) y0 = s.x;
            else
                y[k2] = make_double2(2.0 * s.x, 2.0 * s.y);
        }
#pragma unroll
        for (int b = 0; b <= h; ++b)
        {
            // points n = R2 a + R1 b and R2 a - R1 b (mod P)
            const int n = (R2 * a + R1 * b) % P, m = (R2 * a + R1 * (R2 - b)) % P;
            const int i0 = n == P - 1 ? 0 : n + 1, i1 = m == P - 1 ? 0 : m + 1;
            if (i0 >= W && i1 >= W) continue;
            double C = y0, D = 0.0;
#pragma unroll
            for (int k2 = 1; k2 <= h; ++k2)
            {
                C = fma(kRoots<R2>.c[(b * k2) % R2], y[k2].x, C);
                if (b > 0) D = fma(kRoots<R2>.s[(b * k2) % R2], y[k2].y, D);
            }
            if (i0 < W) acc[i0 < W ? i0 : 0] = C - D;
            if (b > 0 && i1 < W) acc[i1 < W ? i1 : 0] = C + D;
        }
    }
    dst += c * fcs + ji;
    if (lo >= 0)
    {
        double* d = dst + (size_t)lo * G::N3;
        double  old[N];
#pragma unroll
        for (int z = 0; z < N; ++z) old[z] = d[z * G::NN];
#pragma unroll
        for (int z = 0; z < N; ++z) d[z * G::NN] = fma(scale, acc[z], old[z]);
    }
    if (hi >= 0)
    {
        double* d = dst + (size_t)hi * G::N3;
        double  old[N];
#pragma unroll
        for (int z = 0; z < N; ++z) old[z] = d[z * G::NN];
#pragma unroll
        for (int z = 0; z < N; ++z) d[z * G::NN] = fma(scale, acc[E + z], old[z]);
    }
}

// ---------------------------------------------------------------------------
// Kernel spectra (once per block size)
// ---------------------------------------------------------------------------
// One leg of the 14 kernel blocks, out index [o][kz][y or qy][x or qx] built up
// axis by axis: AXIS 0 real z to kz, 1 y to qy, 2 x to qx (stored [qx][qy]).
template<int N, int AXIS>
__global__ __launch_bounds__(kLineThreads) void k_parent_ghat_leg(
    const double* __restrict__ real, const double2* __restrict__ in, double2* __restrict__ out)
{
    using G = Par<N>;
    constexpr int      P = G::P;
    __shared__ double2 tab[P];
    for (int j = threadIdx.x; j < P; j += kLineThreads)
    {
        double s, c;
        sincospi(2.0 * j / P, &s, &c);
        tab[j] = make_double2(c, s);
    }
    __syncthreads();
    const long q = (long)blockIdx.x * kLineThreads + threadIdx.x;
    if (q >= 14L * G::NF) return;
    const int  o = (int)(q / G::NF), f = (int)(q - (long)o * G::NF);
    const int  kz = f / G::PP, hi = (f / P) % P, lo = f % P;
    int        k = kz;
    if (AXIS > 0)
    {
        const int qq = AXIS == 1 ? hi : lo;  // q = k2 R1 + k1 of the leg's axis
        for (k = 0; k % G::R1 != qq % G::R1 || k % G::R2 != qq / G::R1;) ++k;
    }
    double2 s = make_double2(0.0, 0.0);
    for (int m = 0; m < P; ++m)
    {
        const double2 w = tab[k * m % P];
        double2       a;
        if (AXIS == 0) a = make_double2(real[(((long)o * P + m) * P + hi) * P + lo], 0.0);
        else
            a = in[(long)o * G::NF + (long)kz * G::PP + (AXIS == 1 ? m * P + lo : hi * P + m)];
        s.x += a.x * w.x + a.y * w.y;
        s.y += a.y * w.x - a.x * w.y;
    }
    if (AXIS < 2) out[(long)o * G::NF + f] = s;
    else
        out[spec_at(kz * G::PP + lo * P + hi, 0, o, 14)] = s;
}

// ---------------------------------------------------------------------------
// Launches
// ---------------------------------------------------------------------------
inline unsigned blocks_of(long total, int per) { return (unsigned)((total + per - 1) / per); }

// With FP32 spectra the first kz planes are FP64 all the same.  The low
// frequencies are the ones that count: the kernel falls off with the square
// of the frequency, and the rounding of one value near zero frequency reaches the
// whole parent in phase.  18 trees of 73 to 4290 blocks and three components each,
// error against FP64 as a multiple of that of block transforms (mean, largest; the
// coarser levels' part taken out as far as spectra() does): no plane 0.41,
// 1.4; two 0.14, 0.9; three 0.11, 1.3.  4290 blocks, three components: 9.69, 9.74
// and 9.79 ms.
constexpr int kFinePlanes = 2;

constexpr size_t round256(size_t b) { return (b + 255) / 256 * 256; }

// Where a pass keeps its spectra and columns, for ns source and nt target
// parents (times components), in bytes from the start of its scratch; planes
// from `fine` on are FP32.  All planes in one round: the columns of the forward
// legs lie where the target spectra come later, those of the inverse legs
// where the source spectra were.  In rounds of nz planes: the inverse legs'
// columns apart, since the last leg needs all planes; the forward z leg runs
// again every round.
template<class G>
struct Layout
{
    int    nz = 0;  // planes a round; 0: does not fit
    size_t mid_s = 0, mid_t = 0, sspec = 0, tspec = 0, bytes = 0;

    static Slice slice(int z0, int nz, int fine)
    {
        const int z1 = std::min(z0 + nz, G::H), zl = std::min(std::max(z0, fine), z1);
        auto      first = [](int z) { return z * G::PP / 64; };
        auto      count = [&](int a, int b) { return a < b ? (b * G::PP + 63) / 64 - first(a) : 0; };
        return Slice{z0, z1 - z0, zl, first(z0), count(z0, zl), first(zl), count(zl, z1)};
    }
    Layout(long ns, long nt, int fine, int planes) : nz(planes)
    {
        size_t line = 0;  // bytes of a parent
        for (int z0 = 0; z0 < G::H; z0 += nz)
        {
            const Slice sl = slice(z0, nz, fine);
            line = std::max(line, 64 * (sl.nchunk * sizeof(double2) + sl.nchunkf * sizeof(float2)));
        }
        const size_t S = round256(ns * line), T = round256(nt * line);
        const size_t ms = round256((size_t)ns * nz * G::M * G::M * sizeof(double2));
        const size_t mt = round256((size_t)nt * G::H * G::W * G::W * sizeof(double2));
        sspec = nz == G::H ? 0 : mt;
        tspec = mid_s = nz == G::H ? std::max(S, mt) : mt + S;
        bytes = tspec + std::max(T, ms);
    }
    static Layout fit(long ns, long nt, int fine, size_t room)
    {
        Layout l(ns, nt, fine, G::H);
        for (int z = 2; l.bytes > room && z <= G::H; ++z)  // z rounds
            if ((G::H + z - 1) / z < l.nz) l = Layout(ns, nt, fine, (G::H + z - 1) / z);
        if (l.bytes > room) l.nz = 0;
        return l;
    }
};

template<int N>
struct Run
{
    using G = Par<N>;
    using L = Layout<G>;
    template<class T>
    static void pass(hipStream_t s, const ParentPass& p, const double* src, double* dst, double scale, const Batch& b)
    {
        const long ns = (long)p.nsrc * b.k, nt = (long)p.ntgt * b.k;
        const int  fine = fine_planes(sizeof(T) == 4);
        const L    l = L::fit(ns, nt, fine, p.bytes);
        if (l.nz == 0) throw std::logic_error("parent_pass: scratch too small");
        char*    at = static_cast<char*>(p.scratch);
        auto     to = [&](size_t o) { return reinterpret_cast<double2*>(at + o); };
        double2 *mid_s = to(l.mid_s), *mid_t = to(l.mid_t), *sspec = to(l.sspec), *tspec = to(l.tspec);
        // (group, component) pairs a wave: fewer read the kernel values more often, more leave a chunk's
        // sources to L2 for longer (4290 blocks, 2 and 4 pairs: FP64 1.058 and 1.065 ms, with fewer blocks
        // 0.389 and 0.404; FP32, three components, 1.95 and 1.83)
        constexpr int kRun = sizeof(T) == 8 ? 2 : 4;
        const int nseg = (int)std::min(64L, ((long)p.ngroup * b.k + kRun * kMacWaves - 1) / (kRun * kMacWaves));
        const dim3 zgrid(blocks_of(ns * G::M * G::M, kLineThreads)), zthreads(kLineThreads);
        for (int z0 = 0; z0 < G::H; z0 += l.nz)
        {
            const Slice sl = L::slice(z0, l.nz, fine);
            if (l.nz == G::H)
                hipLaunchKernelGGL((k_parent_fwd_z<N, false>), zgrid, zthreads, 0, s, src, b.fstride, p.src_child, p.nsrc,
                    b.k, mid_s, 0, G::H);
            else
                hipLaunchKernelGGL((k_parent_fwd_z<N, true>), zgrid, zthreads, 0, s, src, b.fstride, p.src_child, p.nsrc,
                    b.k, mid_s, sl.z0, sl.nz);
            hipLaunchKernelGGL((k_parent_fwd_plane<N, T>), dim3((unsigned)(ns * sl.nz)), dim3(G::T), 0, s, mid_s, sspec,
                (int)ns, sl);
            hipLaunchKernelGGL(k_parent_mac<T>, dim3((unsigned)((sl.nchunk + sl.nchunkf + 7) / 8 * 8 * nseg)), dim3(64 * kMacWaves), 0,
                s, p.group, p.begin, p.entries, p.ngroup, p.ntgt, p.nsrc, b.k, p.ghat, sspec, tspec, sl, nseg);
            hipLaunchKernelGGL(
                (k_parent_inv_plane<N, T>), dim3((unsigned)(nt * sl.nz)), dim3(G::T), 0, s, tspec, mid_t, (int)nt, sl);
        }
        hipLaunchKernelGGL(k_parent_inv_z<N>, dim3(blocks_of(nt * 4 * G::NN, kLineThreads)), dim3(kLineThreads), 0, s,
            mid_t, p.tgt_child, p.ntgt, b.k, dst, b.fstride,
            scale / ((double)G::P * G::P * G::P));
    }
    static constexpr int fine_planes(bool fp32) { return fp32 ? kFinePlanes : G::H; }
    static size_t bytes(long ns, long nt, bool fp32, size_t room)
    {
        const int fine = fine_planes(fp32);
        const L   l = room ? L::fit(ns, nt, fine, room) : L(ns, nt, fine, G::H);
        return l.nz ? l.bytes : 0;
    }
    static void spectra(hipStream_t s, const double* sample, double2* a, double2* b, double2* ghat)
    {
        const dim3 grid(blocks_of(14L * G::NF, kLineThreads)), block(kLineThreads);
        hipLaunchKernelGGL((k_parent_ghat_leg<N, 0>), grid, block, 0, s, sample, (const double2*)nullptr, a);
        hipLaunchKernelGGL((k_parent_ghat_leg<N, 1>), grid, block, 0, s, (const double*)nullptr, a, b);
        hipLaunchKernelGGL((k_parent_ghat_leg<N, 2>), grid, block, 0, s, (const double*)nullptr, b, ghat);
    }
    static ParentGeo geo() { return ParentGeo{G::M, G::W, G::P, G::H, G::NCH * 64}; }
};

template<class F>
auto on_n(int n, F&& f)
{
    switch (n)
    {
        case 8: return f(Run<8>{});
        case 10: return f(Run<10>{});
        case 12: return f(Run<12>{});
        case 16: return f(Run<16>{});
        case 18: return f(Run<18>{});
        default: throw std::runtime_error("unsupported block size n (supported: 8, 10, 12, 16, 18)");
    }
}

}  // namespace

namespace launch {

ParentGeo parent_geo(int n)
{
    return on_n(n, [](auto r) { return decltype(r)::geo(); });
}
void parent_pass(hipStream_t s, int n, int prec, const ParentPass& p, const double* src, double* dst, double scale,
    const Batch& b)
{
    if (p.nsrc <= 0 || p.ntgt <= 0) return;
    const ParentGeo g = parent_geo(n);
    if ((long)p.nsrc * b.k * g.H > 0x7fffffffL || (long)p.ntgt * b.k * g.H > 0x7fffffffL)
        throw std::invalid_argument("parent_pass: too many parents for one launch");
    on_n(n, [&](auto r) {
        using R = decltype(r);
        if (prec == 0) R::template pass<double>(s, p, src, dst, scale, b);
        else
            R::template pass<float>(s, p, src, dst, scale, b);
    });
}
size_t parent_bytes(int n, int prec, long nsrc, long ntgt, size_t room)
{
    return on_n(n, [&](auto r) { return decltype(r)::bytes(nsrc, ntgt, prec != 0, room); });
}
void parent_spectra(hipStream_t s, int n, const double* sample, double2* a, double2* b, double2* ghat)
{
    on_n(n, [&](auto r) { decltype(r)::spectra(s, sample, a, b, ghat); });
}

}  // namespace launch
}  // namespace iblgf_amd
