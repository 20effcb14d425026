// The three-dimensional FP64 transforms of the field spectrum and its Monte Carlo covariance
// (spectrum.f90:344-567, 569-734), for the compile-time sizes.  Only the shells' summed |.|^2 are
// wanted, so the passes at both ends take their neighbours in: the first pass along an axis makes
// its input itself (random modes, the masked field, the window), the mask of a realisation is
// applied between its forward and backward transform along z, in registers, and the last pass (x)
// writes |.|^2 of kx and -kx added, N/2 + 1 reals a row, in place of the N complex values.  Modes
// beyond the last bin are a fifth of the rows (ky, kz): those rows are neither transformed along x
// nor read or written by the y pass.
//
// A realisation moves 7.5 N^3 complex values (120 B a site) instead of 14.5: at 256^3 790 -> 520 us (modes and x 166,
// forward y 71, z and mask 113, backward y 73, x and folding 62, binning 37), at 512^3 7.9 -> 5.1
// ms; a field spectrum at 512^3 9.9 -> 8.1 ms.  The y and x passes run at the rate of a copy, the
// modes at the rate of their FP64 logarithm, sine and cosine, the z pass, two transforms on one read,
// at 60 % of a copy.
#include "axg_internal.h"
#include "fft_p2.h"

namespace axg {

namespace {

// Is the row (ky, kz) within the last bin's |n|^2?
template <int N> __device__ __forceinline__ bool row_in(int ky, int kz, int64_t n2max)
{
    const int ny = wrapn(ky, N), nz = wrapn(kz, N);
    return (int64_t)ny * ny + (int64_t)nz * nz <= n2max;
}

// 13^(13 * 4 * n) mod 2^64: what n modes of four draws each advance the MCG59 stream by.
constexpr uint64_t mcg59_step(int n)
{
    uint64_t r = 1;
    for (int i = 0; i < 4 * n; i++) r *= MCG59_A;
    return r;
}

// Rows of one Monte Carlo realisation (spectrum.f90:592-641), transformed along x (FORWARD): mode k gets
// a unit complex Gaussian times sigma[b] of its spectrum bin b, or 0 outside the bins.  The
// Gaussian of mode k in realisation iter (1-based): from the reference's stream, draws
// pos + 4 N^3 (iter - 1) + 4 k .. +3 (every mode draws, binned or not, as there; a thread's eight
// modes are N/8 apart, so it jumps once and steps by a constant); otherwise Philox4x32-10 keyed by
// the seed, counter = (mode index, 'cov ', iter).
template <int N>
__global__ void __launch_bounds__(p2_rows_per_block<N>() * (N / 8))
    spec_modes_x_kernel(Draws dr, int iter, const uint16_t* __restrict__ bin_of_n2, int64_t n2max,
                        const double* __restrict__ sigma, double2* __restrict__ out, const double2* __restrict__ tw)
{
    constexpr int TPT = N / 8, RB = p2_rows_per_block<N>();
    constexpr int64_t NN = (int64_t)N * N, n3 = NN * N;
    __shared__ double2 s[RB * N];
    const int rr = threadIdx.x / TPT, j0 = threadIdx.x % TPT;
    const int64_t row = (int64_t)blockIdx.x * RB + rr;
    const int kz = (int)(row / N), ky = (int)(row - (int64_t)kz * N);
    const bool active = row < NN && row_in<N>(ky, kz, n2max);
    if (!__syncthreads_or(active)) return;
    double2 v[8];
    if (active) {
#pragma clang fp contract(off)
        const uint64_t seed = (uint64_t)dr.k0 | ((uint64_t)dr.k1 << 32);
        const int ny = wrapn(ky, N), nz = wrapn(kz, N);
        uint64_t xs = dr.mcg ? mcg59_jump(dr.x0, dr.pos + 4 * (uint64_t)n3 * (iter - 1) + 4 * (uint64_t)(row * N + j0)) : 0;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int kx = j0 + e * TPT, nx = wrapn(kx, N);
            const int b = bin_of_n2[(int64_t)nx * nx + (int64_t)ny * ny + (int64_t)nz * nz];
            v[e] = double2{0, 0};
            if (b > 0) {
                double g1, g2;
                if (dr.mcg) {
                    uint64_t x = xs;
                    g1 = mcg59_gauss(x);
                    g2 = mcg59_gauss(x);
                } else {
                    unit_gauss(seed, 0x636f7620u, (uint32_t)iter, (uint64_t)(row * N + kx), g1, g2);
                }
                const double sg = sigma[b - 1];
                v[e] = double2{g1 * sg, g2 * sg};
            }
            xs = (xs * mcg59_step(TPT)) & MCG59_MASK;
        }
    }
    fft_p2_if<double, N, -1>(active, v, j0, s + rr * N, 1, 0, p2_load_twiddles<double, N, -1>(j0, tw));
    if (active) {
#pragma unroll
        for (int e = 0; e < 8; e++) out[row * N + j0 + e * TPT] = v[e];
    }
}

// Transform along y, in place: block = one plane kz and a tile of x columns.  LIM 1: rows beyond n2max
// are not read (they are zero); LIM 2: they are not written (nothing reads them).
template <int N, int SIGN, int LIM>
__global__ void __launch_bounds__((p2_tx<double, N>() * (N / 8))) spec_y_kernel(double2* __restrict__ data, int64_t n2max,
                                                                          const double2* __restrict__ tw)
{
    constexpr int TX = p2_tx<double, N>(), TPT = N / 8;
    __shared__ double2 s[N * TX];
    const int b = threadIdx.x % TX, j0 = threadIdx.x / TX, kz = blockIdx.y;
    const int col = blockIdx.x * TX + b;
    const bool ok = col < N;
    double2* base = data + (int64_t)kz * N * N + col;
    double2 v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const int ky = j0 + e * TPT;
        v[e] = ok && (LIM != 1 || row_in<N>(ky, kz, n2max)) ? base[(int64_t)ky * N] : double2{0, 0};
    }
    fft_p2<double, N, SIGN>(v, j0, s, TX, b, p2_load_twiddles<double, N, SIGN>(j0, tw));
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const int ky = j0 + e * TPT;
        if (ok && (LIM != 2 || row_in<N>(ky, kz, n2max))) base[(int64_t)ky * N] = v[e];
    }
}

// The mask as the z transforms read it: bit x % 8 of bits[y][x / 8][z], so that a tile of columns finds its
// mask in N consecutive bytes.  (Read from the flags themselves, eight bytes of each 128-byte line,
// it is as much traffic as the tile.)  One thread per byte, z fastest across the rows it reads.
__global__ void __launch_bounds__(256) spec_mask_bits_kernel(int N, const int8_t* __restrict__ flags, uint8_t* __restrict__ bits)
{
    const int nx8 = (N + 7) / 8;
    const int xt = blockIdx.x * 32 + threadIdx.x % 32, z = blockIdx.y * 8 + threadIdx.x / 32, y = blockIdx.z;
    if (xt >= nx8 || z >= N) return;
    const int8_t* f = flags + ((int64_t)z * N + y) * N + 8 * xt;
    uint8_t m = 0;
    for (int k = 0; k < 8 && 8 * xt + k < N; k++) m |= (uint8_t)(((f[k] >> 2) & 1) << k);
    bits[((int64_t)y * nx8 + xt) * N + z] = m;
}

// A realisation's transforms along z: FORWARD, the mask's cells zeroed, BACKWARD; in place, one read and
// one write of the array for what took three passes.  Block = one y and a tile of x columns.
template <int N>
__global__ void __launch_bounds__((p2_tx<double, N>() * (N / 8))) spec_z_mask_kernel(double2* __restrict__ data,
                                                                               const uint8_t* __restrict__ bits,
                                                                               const double2* __restrict__ tw)
{
    constexpr int TX = p2_tx<double, N>(), TPT = N / 8;
    constexpr int64_t NN = (int64_t)N * N;
    __shared__ double2 s[N * TX];
    const int b = threadIdx.x % TX, j0 = threadIdx.x / TX;
    const int col = blockIdx.x * TX + b;
    const bool ok = col < N;
    const int64_t i0 = (int64_t)blockIdx.y * N + col;
    const uint8_t* mb = bits + ((int64_t)blockIdx.y * ((N + 7) / 8) + (ok ? col / 8 : 0)) * N;
    double2 v[8];
    int m = 0;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        v[e] = ok ? data[i0 + (j0 + e * TPT) * NN] : double2{0, 0};
        m |= ((mb[j0 + e * TPT] >> (col % 8)) & 1) << e;
    }
    fft_p2<double, N, -1>(v, j0, s, TX, b, P2TwTable<double, N, -1>{tw, j0});
#pragma unroll
    for (int e = 0; e < 8; e++)
        if ((m >> e) & 1) v[e] = double2{0, 0};
    fft_p2<double, N, +1>(v, j0, s, TX, b, P2TwTable<double, N, +1>{tw, j0});
    if (ok) {
#pragma unroll
        for (int e = 0; e < 8; e++) data[i0 + (j0 + e * TPT) * NN] = v[e];
    }
}

// BACKWARD transform along z of (mask ? 0 : pi), or of (mask ? 0 : fill) for the window, into out.
template <typename T, bool COMP, int N>
__global__ void __launch_bounds__((p2_tx<double, N>() * (N / 8))) spec_z_field_kernel(
    const typename V2<T>::type* __restrict__ pi, const short2* __restrict__ cpi, const int8_t* __restrict__ flags,
    double fill, int use_pi, double2* __restrict__ out, const double2* __restrict__ tw)
{
    constexpr int TX = p2_tx<double, N>(), TPT = N / 8;
    constexpr int64_t NN = (int64_t)N * N;
    __shared__ double2 s[N * TX];
    const int b = threadIdx.x % TX, j0 = threadIdx.x / TX;
    const int col = blockIdx.x * TX + b;
    const bool ok = col < N;
    const int64_t i0 = (int64_t)blockIdx.y * N + col;
    double2 v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const int64_t i = i0 + (j0 + e * TPT) * NN;
        v[e] = double2{0, 0};
        if (ok) {
            const bool masked = flags[i] & 4;
            if (use_pi) v[e] = ldf<T, COMP>(pi, cpi, i);
            else v[e].x = fill;
            if (masked) v[e] = double2{0, 0};
        }
    }
    fft_p2<double, N, +1>(v, j0, s, TX, b, p2_load_twiddles<double, N, +1>(j0, tw));
    if (ok) {
#pragma unroll
        for (int e = 0; e < 8; e++) out[i0 + (j0 + e * TPT) * NN] = v[e];
    }
}

// BACKWARD transform along x of the rows within n2max and their folded power (SpecPair), N/2 + 1 reals at the
// beginning of the row's own N complex values.
template <int N>
__global__ void __launch_bounds__(p2_rows_per_block<N>() * (N / 8))
    spec_fold_x_kernel(double2* __restrict__ data, int64_t n2max, double amp, const double2* __restrict__ tw)
{
    constexpr int TPT = N / 8, RB = p2_rows_per_block<N>();
    __shared__ double2 s[RB * N];
    const int rr = threadIdx.x / TPT, j0 = threadIdx.x % TPT;
    const int64_t row = (int64_t)blockIdx.x * RB + rr;
    const int kz = (int)(row / N), ky = (int)(row - (int64_t)kz * N);
    const bool active = row < (int64_t)N * N && row_in<N>(ky, kz, n2max);
    if (!__syncthreads_or(active)) return;
    double2* base = data + (active ? row : 0) * N;
    double2* sr = s + rr * N;
    double2 v[8];
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = active ? base[j0 + e * TPT] : double2{0, 0};
    fft_p2_if<double, N, +1>(active, v, j0, sr, 1, 0, p2_load_twiddles<double, N, +1>(j0, tw));
#pragma unroll
    for (int e = 0; e < 8; e++) sr[j0 + e * TPT] = v[e];
    __syncthreads();
    if (active) {
#pragma unroll
        for (int i = 0; i < 5; i++) {
            const int j = j0 + i * TPT;
            if (j > N / 2) continue;
            SpecPair<false> p;
            p.load(sr, N, j);
            reinterpret_cast<double*>(base)[j] = p.power(amp);
        }
    }
}

}  // namespace

bool launch_spec_modes_x(hipStream_t s, int N, const Draws& dr, int iter, const uint16_t* bin_of_n2, int64_t n2max,
                         const double* sigma, double2* out, const double2* tw)
{
    const bool done = p2_dispatch(N, [&]<int NN>() {
        constexpr int RB = p2_rows_per_block<NN>();
        hipLaunchKernelGGL(spec_modes_x_kernel<NN>, dim3((NN * NN + RB - 1) / RB), dim3(RB * (NN / 8)), 0, s, dr, iter,
                           bin_of_n2, n2max, sigma, out, tw);
    });
    if (done) AXG_HIP(hipGetLastError());
    return done;
}

void launch_spec_y(hipStream_t s, int N, double2* data, int sign, int lim, int64_t n2max, const double2* tw)
{
    const bool done = p2_dispatch(N, [&]<int NN>() {
        constexpr int TX = p2_tx<double, NN>();
        const dim3 grid((NN + TX - 1) / TX, NN), blk(TX * (NN / 8));
        if (sign < 0) hipLaunchKernelGGL((spec_y_kernel<NN, -1, 1>), grid, blk, 0, s, data, n2max, tw);
        else if (lim) hipLaunchKernelGGL((spec_y_kernel<NN, +1, 2>), grid, blk, 0, s, data, n2max, tw);
        else hipLaunchKernelGGL((spec_y_kernel<NN, +1, 0>), grid, blk, 0, s, data, n2max, tw);
    });
    if (!done) throw Error(AXG_EINVAL, "spectrum passes need a compile-time size");
    AXG_HIP(hipGetLastError());
}

size_t spec_mask_bytes(int N) { return (size_t)N * ((N + 7) / 8) * N; }

void launch_spec_mask_bits(hipStream_t s, int N, const int8_t* flags, uint8_t* bits)
{
    hipLaunchKernelGGL(spec_mask_bits_kernel, dim3(((N + 7) / 8 + 31) / 32, (N + 7) / 8, N), dim3(256), 0, s, N, flags, bits);
    AXG_HIP(hipGetLastError());
}

void launch_spec_z_mask(hipStream_t s, int N, double2* data, const uint8_t* bits, const double2* tw)
{
    const bool done = p2_dispatch(N, [&]<int NN>() {
        constexpr int TX = p2_tx<double, NN>();
        hipLaunchKernelGGL(spec_z_mask_kernel<NN>, dim3((NN + TX - 1) / TX, NN), dim3(TX * (NN / 8)), 0, s, data, bits, tw);
    });
    if (!done) throw Error(AXG_EINVAL, "spectrum passes need a compile-time size");
    AXG_HIP(hipGetLastError());
}

template <typename T, bool COMP>
bool launch_spec_z_field(hipStream_t s, int N, const void* pi, const void* cpi, const int8_t* flags, double fill, bool use_pi,
                         double2* out, const double2* tw)
{
    using T2 = typename V2<T>::type;
    const bool done = p2_dispatch(N, [&]<int NN>() {
        constexpr int TX = p2_tx<double, NN>();
        hipLaunchKernelGGL((spec_z_field_kernel<T, COMP, NN>), dim3((NN + TX - 1) / TX, NN), dim3(TX * (NN / 8)), 0, s,
                           (const T2*)pi, (const short2*)cpi, flags, fill, use_pi ? 1 : 0, out, tw);
    });
    if (done) AXG_HIP(hipGetLastError());
    return done;
}
template bool launch_spec_z_field<double, false>(hipStream_t, int, const void*, const void*, const int8_t*, double, bool,
                                                 double2*, const double2*);
template bool launch_spec_z_field<float, false>(hipStream_t, int, const void*, const void*, const int8_t*, double, bool,
                                                double2*, const double2*);
template bool launch_spec_z_field<float, true>(hipStream_t, int, const void*, const void*, const int8_t*, double, bool,
                                               double2*, const double2*);

void launch_spec_fold_x(hipStream_t s, int N, double2* data, int64_t n2max, double amp, const double2* tw)
{
    const bool done = p2_dispatch(N, [&]<int NN>() {
        constexpr int RB = p2_rows_per_block<NN>();
        hipLaunchKernelGGL(spec_fold_x_kernel<NN>, dim3((NN * NN + RB - 1) / RB), dim3(RB * (NN / 8)), 0, s, data, n2max, amp,
                           tw);
    });
    if (!done) throw Error(AXG_EINVAL, "spectrum passes need a compile-time size");
    AXG_HIP(hipGetLastError());
}

}  // namespace axg
