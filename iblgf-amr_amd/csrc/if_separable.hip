// Neighbour-only integrating-factor pass as separable sums.
//
// The factor's point kernel is a product of one-dimensional ones,
// E(x, y, z) = iv[|x|] iv[|y|] iv[|z|], and a pass without far field sums a
// target block over the 27 neighbour blocks (Fmm::apply with the integrating
// factor, include/iblgf/fmm/fmm.hpp:729-870 with non-Laplace kernels), a
// range that is a product as well.  So the pass is three one-dimensional sums
// over at most three blocks each, exactly, without transforms: z over a
// block's interior columns into scratch, then y and x per target.  A target
// of n = 18 costs 1.2 million fused multiply-adds and about 130 KB of traffic;
// the transforms it replaces cost 7.5 million (forward, inverse, 27 spectra)
// and 2.2 MB.  Three face components on a 1422-block adaptive tree of 16^3
// cells: the solve took 3.32 ms through the transforms and takes 0.61 ms.
#include "kernels.hpp"

#include <stdexcept>

namespace iblgf_amd {
namespace {

// acc[k] += sum_a iv[|E O + a + 1 - k|] v_a for the E interior points of the
// neighbour at offset O on the leg's axis and the N points of the target
// (boundary ring included).  The at most 2 E + 1 values of iv in use are read
// at constant indices, the same for the whole wave: they sit in scalar
// registers and no matrix is loaded.
template<int N, int O, class Load>
__device__ inline void band(const double* __restrict__ iv, double (&acc)[N], Load&& load)
{
    constexpr int E = N - 2;
#pragma unroll
    for (int a = 0; a < E; ++a)
    {
        const double v = load(a);
#pragma unroll
        for (int k = 0; k < N; ++k)
        {
            constexpr int base = E * O + 1;
            const int     d = base + a - k;
            acc[k] = fma(iv[d < 0 ? -d : d], v, acc[k]);
        }
    }
}

constexpr int kSepThreads = 256;

// z leg: mid[pos][k][y][x] = sum over the three blocks zent[3 pos ..] (-1:
// none) below, at and above position pos.  One thread per interior column;
// neighbouring threads take neighbouring x, so every load and store of a wave
// covers whole runs of a row.
template<int N>
__global__ __launch_bounds__(kSepThreads) void k_if_z(const double* __restrict__ src, double* __restrict__ mid,
    const int* __restrict__ zent, int npos, const double* __restrict__ iv, long fcs, long mcs)
{
    constexpr int E = N - 2, EE = E * E, NN = N * N, N3 = N * NN;
    const int     q = xcd_item(blockIdx.x, gridDim.x) * kSepThreads + threadIdx.x;
    const int     pos = q / EE, col = q - pos * EE;
    if (pos >= npos) return;
    src += blockIdx.y * fcs + NN + (col / E + 1) * N + col % E + 1;
    mid += blockIdx.y * mcs + (size_t)pos * (N * EE) + col;
    double acc[N];
#pragma unroll
    for (int k = 0; k < N; ++k) acc[k] = 0.0;
    const int lo = zent[3 * pos], at = zent[3 * pos + 1], hi = zent[3 * pos + 2];
    if (lo >= 0) band<N, -1>(iv, acc, [&](int a) { return src[(size_t)lo * N3 + a * NN]; });
    if (at >= 0) band<N, 0>(iv, acc, [&](int a) { return src[(size_t)at * N3 + a * NN]; });
    if (hi >= 0) band<N, 1>(iv, acc, [&](int a) { return src[(size_t)hi * N3 + a * NN]; });
#pragma unroll
    for (int k = 0; k < N; ++k) mid[k * EE] = acc[k];
}

// y and x legs of one target (and component): dst[target] += the sum over
// the nine positions ent[1 + (ox + 1) + 3 (oy + 1)] (-1: none).  Per ox the y
// leg runs on N E threads from scratch into LDS (index x, then z, y), the x
// leg on N N threads from LDS into registers; the block goes out through LDS
// so that its read-add-write is contiguous.
template<int N>
constexpr int sep_threads() { return (N * N + 63) / 64 * 64; }

template<int N>
__global__ __launch_bounds__(sep_threads<N>()) void k_if_yx(const double* __restrict__ mid, double* __restrict__ dst,
    const int* __restrict__ entries, int ntgt, const double* __restrict__ iv, long mcs, long fcs)
{
    constexpr int E = N - 2, EE = E * E, NN = N * N, N3 = N * NN, T = sep_threads<N>();
    // odd rows: the y leg's 64-bit stores, a stride of one row apart, meet different banks
    constexpr int     ROW = NN + 1;
    constexpr int     kBuf = E * ROW > N3 ? E * ROW : N3;
    __shared__ double buf[kBuf];
    const int         item = xcd_item(blockIdx.x, gridDim.x);
    if (item >= ntgt) return;  // the whole workgroup
    const int*        ent = entries + 10 * item;
    const int         l = threadIdx.x, z = l / E, x = l - z * E;
    mid += blockIdx.y * mcs + z * EE + x;
    double out[N];
#pragma unroll
    for (int k = 0; k < N; ++k) out[k] = 0.0;
#pragma unroll 1
    for (int ox = 0; ox < 3; ++ox)
    {
        const int lo = ent[1 + ox], at = ent[4 + ox], hi = ent[7 + ox];
        if (lo < 0 && at < 0 && hi < 0) continue;  // the same for the whole workgroup
        if (l < N * E)
        {
            double acc[N];
#pragma unroll
            for (int k = 0; k < N; ++k) acc[k] = 0.0;
            if (lo >= 0) band<N, -1>(iv, acc, [&](int a) { return mid[(size_t)lo * (N * EE) + a * E]; });
            if (at >= 0) band<N, 0>(iv, acc, [&](int a) { return mid[(size_t)at * (N * EE) + a * E]; });
            if (hi >= 0) band<N, 1>(iv, acc, [&](int a) { return mid[(size_t)hi * (N * EE) + a * E]; });
#pragma unroll
            for (int k = 0; k < N; ++k) buf[x * ROW + z * N + k] = acc[k];
        }
        __syncthreads();
        if (l < NN)
        {
            auto line = [&](int a) { return buf[a * ROW + l]; };
            if (ox == 0) band<N, -1>(iv, out, line);
            else if (ox == 1) band<N, 0>(iv, out, line);
            else
                band<N, 1>(iv, out, line);
        }
        __syncthreads();
    }
    if (l < NN)
    {
#pragma unroll
        for (int k = 0; k < N; ++k) buf[l * N + k] = out[k];
    }
    __syncthreads();
    dst += blockIdx.y * fcs + (size_t)ent[0] * N3;
    for (int q = l; q < N3; q += T) dst[q] += buf[q];
}

template<int N>
void run(hipStream_t s, const double* src, double* mid, double* dst, const int* zent, int npos, const int* ent,
    int ntgt, const double* iv, const Batch& b, long mcs)
{
    const long cols = (long)npos * (N - 2) * (N - 2);
    hipLaunchKernelGGL(k_if_z<N>, dim3(xcd_grid((cols + kSepThreads - 1) / kSepThreads), b.k), dim3(kSepThreads), 0,
        s, src, mid, zent, npos, iv, b.fstride, mcs);
    hipLaunchKernelGGL(k_if_yx<N>, dim3(xcd_grid(ntgt), b.k), dim3(sep_threads<N>()), 0, s, mid, dst, ent, ntgt, iv, mcs,
        b.fstride);
}

}  // namespace

namespace launch {

void if_separable(hipStream_t s, int n, const double* src, double* mid, double* dst, const int* zent, int npos,
    const int* ent, int ntgt, const double* iv, const Batch& b, long mid_stride)
{
    if (npos <= 0 || ntgt <= 0) return;
    if (mid_stride < if_mid_size(n) * npos && b.k > 1) throw std::invalid_argument("if_separable: scratch stride");
    switch (n)
    {
        case 8: run<8>(s, src, mid, dst, zent, npos, ent, ntgt, iv, b, mid_stride); break;
        case 10: run<10>(s, src, mid, dst, zent, npos, ent, ntgt, iv, b, mid_stride); break;
        case 12: run<12>(s, src, mid, dst, zent, npos, ent, ntgt, iv, b, mid_stride); break;
        case 16: run<16>(s, src, mid, dst, zent, npos, ent, ntgt, iv, b, mid_stride); break;
        case 18: run<18>(s, src, mid, dst, zent, npos, ent, ntgt, iv, b, mid_stride); break;
        default: throw std::runtime_error("unsupported block size n (supported: 8, 10, 12, 16, 18)");
    }
}

}  // namespace launch
}  // namespace iblgf_amd
