// DCT-II / its inverse along chosen axes of batched 3-D complex64 volumes, and the L1
// soft-threshold prox in the DCT domain (ProximalL1DCT, python/python/hastypy/base/
// proximal.py:134-183, which calls cupyx.scipy.fft.dctn / idctn with norm=None):
//   dct:  y_k = 2 sum_n x_n cos(pi k (2n + 1) / (2N))
//   idct: x_n = (1 / 2N) (y_0 + 2 sum_{k>=1} y_k cos(pi k (2n + 1) / (2N)))
// Each axis pass is a real N x N matrix (N <= 512) applied to every line with
// v_mfma_f32_16x16x4f32. The matrix is even or odd about the middle of n, so with
//   E_n = x_n + x_{N-1-n},  O_n = x_n - x_{N-1-n}   (n < N/2)
// y_{2j} needs E alone and y_{2j+1} O alone (and back: x_n, x_{N-1-n} = a_n +- b_n, a from
// the even and b from the odd frequencies): two products of half the size, a quarter of
// the multiply-adds each.
//
// A workgroup stages the lines of 32 complex columns in LDS as the two half-size parts
// (formed while loading), multiplies, and writes the lines back; each wave owns the same
// row tile of both parts. The prox runs the last forward axis, the threshold and the
// first inverse axis in one pass (the strided axis' results are already split by parity),
// so it makes five passes over the volumes instead of seven. 5 volumes of 96 x 128 x 128:
// 1065 us with one thread per output reading the matrix from L2 and a matrix built,
// allocated and freed per axis and call; 231 us here (a pass of 126 MB: 39 us, fused
// 67 us; the HBM rate of a copy gives 24).
#include <cmath>
#include <map>
#include <mutex>
#include <tuple>

#include "common.hpp"
#include "toeplitz.hpp"

namespace hasty_hip {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kDctThreads = 256;
constexpr int kDctCols = 32;              // complex lines per workgroup
constexpr int kColStride = 2 * kDctCols + 16;  // floats per LDS row of the strided form: the four
                                               // rows one MFMA operand reads start 16 banks apart

// Matrix tiles in MFMA operand order, rt = ceil(ceil(N/2) / 16) tiles per side: part 0 maps
// E to the even (or, inverse, the even frequencies to a), part 1 O to the odd ones (b).
// Entry (part, row tile i, k group q, lane, u): row 16 i + (lane & 15), column
// 16 q + 4 u + (lane >> 4); zero outside the matrix, so padded rows and columns stay zero.
__global__ void dct_tiles_kernel(float* tiles, int N, int rt, int inverse)
{
    const int e = blockIdx.x * kDctThreads + threadIdx.x;
    if (e >= 2 * rt * rt * 256) return;
    const int u = e & 3, lane = (e >> 2) & 63, q = (e >> 8) % rt, i = (e >> 8) / rt % rt, part = (e >> 8) / (rt * rt);
    const int r = 16 * i + (lane & 15), c = 16 * q + 4 * u + (lane >> 4);
    const int n = inverse ? r : c, j = inverse ? c : r;  // sample and half-frequency index
    const int k = 2 * j + part;
    double v = 0.0;
    if (n < (part ? N / 2 : (N + 1) / 2) && k < N) {
        v = 2.0 * cos(M_PI * (double)((int64_t)k * (2 * n + 1) % (4 * N)) / (2.0 * N));
        if (inverse) v *= (k == 0 ? 0.5 : 1.0) / (2.0 * N);
    }
    tiles[e] = (float)v;
}

std::mutex g_tiles_mutex;
// (device, N, inverse), held until the process ends, as the FFT's twiddles are: at most 512 KB
// each, 196 MB if every length of 2 to 512 were used both ways
std::map<std::tuple<int, int, int>, float*> g_tiles;

// The tiles of one transform, built on first use (a graph capture must come after that).
const float* dct_tiles(int N, int inverse, hipStream_t s)
{
    const auto key = std::make_tuple(current_device(), N, inverse);
    std::lock_guard<std::mutex> lock(g_tiles_mutex);
    const auto it = g_tiles.find(key);
    if (it != g_tiles.end()) return it->second;
    const int rt = ((N + 1) / 2 + 15) / 16;
    const int n = 2 * rt * rt * 256;
    float* t = (float*)dev_alloc_table(sizeof(float) * n);
    try {
        hipLaunchKernelGGL(dct_tiles_kernel, dim3((unsigned)ceil_div(n, kDctThreads)), dim3(kDctThreads), 0, s, t, N, rt,
                           inverse);
        check_launch("dct_tiles_kernel");
        HASTY_HIP_CHECK(hipStreamSynchronize(s));
    } catch (...) {
        dev_free(t);
        throw;
    }
    g_tiles[key] = t;
    return t;
}

// acc[w][part][c] += tile row (wave + 4 w) of `part` times the staged data of column tile c:
// the operand of k step (q, u) is X[part][c](16 q + 4 u + lane / 16), through `ld`. SWAP
// puts the data first (rows of the result are data columns, columns matrix rows).
template <int PW, bool SWAP, typename Ld>
__device__ __forceinline__ void dct_multiply(floatx4 (&acc)[PW][2][4], const float* __restrict__ tiles, int rt, Ld ld)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const float4* t4 = reinterpret_cast<const float4*>(tiles) + lane;
#pragma unroll
    for (int w = 0; w < PW; ++w)
#pragma unroll
        for (int part = 0; part < 2; ++part)
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[w][part][c] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (wave >= rt) return;  // fewer row tiles than waves
    for (int q = 0; q < rt; ++q) {
#pragma unroll
        for (int part = 0; part < 2; ++part) {
            float4 m[PW];
#pragma unroll
            for (int w = 0; w < PW; ++w) {
                const int i = min(wave + 4 * w, rt - 1);  // a tile past the end repeats the last one, unused
                m[w] = t4[((part * rt + i) * rt + q) * 64];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                float x[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) x[c] = ld(part, c, 16 * q + 4 * u);
#pragma unroll
                for (int w = 0; w < PW; ++w) {
                    const float mu = u == 0 ? m[w].x : u == 1 ? m[w].y : u == 2 ? m[w].z : m[w].w;
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        acc[w][part][c] =
                            SWAP ? __builtin_amdgcn_mfma_f32_16x16x4f32(x[c], mu, acc[w][part][c], 0, 0, 0)
                                 : __builtin_amdgcn_mfma_f32_16x16x4f32(mu, x[c], acc[w][part][c], 0, 0, 0);
                }
            }
        }
    }
}

// Scale of the soft threshold for the complex value of magnitude^2 m2.
__device__ __forceinline__ float soft_scale(float m2, float thresh)
{
    const float m = sqrtf(m2);
    return m > thresh ? (m - thresh) / m : 0.f;
}

// Lines along a strided axis: the element n of complex column c (c < inner) of slice b is
// data[b * outer + n * inner + c]. A workgroup takes 32 of the columns of all slices (a slice
// of fewer columns would leave it idle: 8 million elements in lines of 128, slices of one
// column, 753 us with a workgroup per slice, 47 us here, 37 us for wide slices either way).
// MODE 0 forward, 1 inverse, 2 forward, threshold, inverse.
template <int PW, int MODE>
__global__ void __launch_bounds__(kDctThreads) dct_strided_kernel(float2* data, const float* __restrict__ fwd,
                                                                  const float* __restrict__ inv, int N, int64_t inner,
                                                                  int64_t outer, int64_t columns, float thresh)
{
    extern __shared__ __align__(16) float lds[];
    const int half = (N + 1) / 2, odd = N / 2, rt = (half + 15) / 16, rows = 16 * rt;
    float* X = lds;  // [2 parts][rows][kColStride]
    const int part_stride = rows * kColStride;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int col = t & 31, r0 = t >> 5;
    const int64_t q = (int64_t)blockIdx.x * kDctCols + col, b = q / inner;
    const bool on = q < columns;
    float2* base = data + b * outer + (q - b * inner);
    auto at = [&](int n) -> float2& { return base[(int64_t)n * inner]; };
    for (int n = r0; n < rows; n += kDctThreads / 32) {
        float2 e = float2{0.f, 0.f}, o = float2{0.f, 0.f};
        if (on && n < half) {
            if (MODE == 1) {
                e = at(2 * n);
                if (n < odd) o = at(2 * n + 1);
            } else {
                e = at(n);
                if (n < odd) {
                    const float2 y = at(N - 1 - n);
                    o = csub(e, y);
                    e = cadd(e, y);
                }
            }
        }
        *reinterpret_cast<float2*>(X + n * kColStride + 2 * col) = e;
        *reinterpret_cast<float2*>(X + part_stride + n * kColStride + 2 * col) = o;
    }
    __syncthreads();
    floatx4 acc[PW][2][4];
    const float* Xl = X + (lane >> 4) * kColStride + (lane & 15);
    auto ld = [&](int part, int c, int k) { return Xl[part * part_stride + k * kColStride + 16 * c]; };
    // accumulator element v: row 16 i + 4 (lane / 16) + v, column 16 c + (lane & 15)
    auto put = [&](bool combine) {
        __syncthreads();  // every wave has read the staged data
#pragma unroll
        for (int w = 0; w < PW; ++w) {
            const int i = wave + 4 * w;
            if (i >= rt) continue;
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    float* d = X + (16 * i + 4 * (lane >> 4) + v) * kColStride + 16 * c + (lane & 15);
                    const float p = acc[w][0][c][v], q = acc[w][1][c][v];
                    d[0] = combine ? p + q : p;
                    d[part_stride] = combine ? p - q : q;
                }
        }
        __syncthreads();
    };
    dct_multiply<PW, false>(acc, MODE == 1 ? inv : fwd, rt, ld);
    if (MODE == 2) {
        // neighbouring lanes hold the real and the imaginary part of one column
#pragma unroll
        for (int w = 0; w < PW; ++w)
#pragma unroll
            for (int part = 0; part < 2; ++part)
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float x = acc[w][part][c][v];
                        const float y = __shfl_xor(x, 1);
                        const bool re = (lane & 1) == 0;
                        const float xr = re ? x : y, xi = re ? y : x;
                        acc[w][part][c][v] = x * soft_scale(xr * xr + xi * xi, thresh);
                    }
        put(false);
        dct_multiply<PW, false>(acc, inv, rt, ld);
    }
    put(MODE != 0);
    for (int n = r0; n < half; n += kDctThreads / 32) {
        if (!on) break;
        const float2 p = *reinterpret_cast<const float2*>(X + n * kColStride + 2 * col);
        const float2 q = *reinterpret_cast<const float2*>(X + part_stride + n * kColStride + 2 * col);
        at(MODE == 0 ? 2 * n : n) = p;
        if (n < odd) at(MODE == 0 ? 2 * n + 1 : N - 1 - n) = q;
    }
}

// LDS floats per line of the contiguous form: the eight lines of an operand's rows start 8
// banks apart.
__host__ __device__ inline int line_stride(int rows) { return 2 * rows + (72 - 2 * rows % 64) % 64; }

// Lines along the contiguous axis; MODE 0 forward, 1 inverse. The data are the first
// operand (rows are line and part re / im), so a lane ends with whole complex values of
// consecutive frequencies or samples and stores them directly.
template <int PW, int MODE>
__global__ void __launch_bounds__(kDctThreads) dct_lines_kernel(float2* data, const float* __restrict__ tiles, int N,
                                                                int64_t nlines)
{
    extern __shared__ __align__(16) float lds[];
    const int half = (N + 1) / 2, odd = N / 2, rt = (half + 15) / 16, rows = 16 * rt;
    const int ls = line_stride(rows);
    const int part_stride = kDctCols * ls;  // [2 parts][32 lines][ls]
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t l0 = (int64_t)blockIdx.x * kDctCols;
    const int nl = (int)min((int64_t)kDctCols, nlines - l0);
    float2* base = data + l0 * N;
    for (int l = wave; l < kDctCols; l += 4) {
        float2* de = reinterpret_cast<float2*>(lds + l * ls);
        float2* dd = reinterpret_cast<float2*>(lds + part_stride + l * ls);
        const float2* line = base + (int64_t)l * N;
        for (int n = lane; n < rows; n += 64) {
            float2 e = float2{0.f, 0.f}, o = float2{0.f, 0.f};
            if (l < nl && n < half) {
                if (MODE == 1) {
                    e = line[2 * n];
                    if (n < odd) o = line[2 * n + 1];
                } else {
                    e = line[n];
                    if (n < odd) {
                        const float2 y = line[N - 1 - n];
                        o = csub(e, y);
                        e = cadd(e, y);
                    }
                }
            }
            de[n] = e;
            dd[n] = o;
        }
    }
    __syncthreads();
    floatx4 acc[PW][2][4];
    // operand row (lane & 15) of row tile c: line 8 c + (lane & 15) / 2, part lane & 1
    const float* Xl = lds + ((lane & 15) >> 1) * ls + 2 * (lane >> 4) + (lane & 1);
    auto ld = [&](int part, int c, int k) { return Xl[part * part_stride + 8 * c * ls + 2 * k]; };
    dct_multiply<PW, true>(acc, tiles, rt, ld);
    // accumulator element v: matrix row j = 16 i + (lane & 15), line 8 c + 2 (lane / 16) + v / 2
#pragma unroll
    for (int w = 0; w < PW; ++w) {
        const int j = 16 * (wave + 4 * w) + (lane & 15);
        if (j >= half) continue;
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int v = 0; v < 4; v += 2) {
                const int l = 8 * c + 2 * (lane >> 4) + v / 2;
                if (l >= nl) continue;
                const float2 p = float2{acc[w][0][c][v], acc[w][0][c][v + 1]};
                const float2 q = float2{acc[w][1][c][v], acc[w][1][c][v + 1]};
                float2* line = base + (int64_t)l * N;
                line[MODE == 0 ? 2 * j : j] = MODE == 0 ? p : cadd(p, q);
                if (j < odd) line[MODE == 0 ? 2 * j + 1 : N - 1 - j] = MODE == 0 ? q : csub(p, q);
            }
    }
}

__global__ void soft_kernel(float2* d, int64_t n, float thresh)
{
    const int64_t i = (int64_t)blockIdx.x * kDctThreads + threadIdx.x;
    if (i >= n) return;
    const float2 v = d[i];
    const float s = soft_scale(v.x * v.x + v.y * v.y, thresh);
    d[i] = float2{v.x * s, v.y * s};
}

// One axis pass; MODE 2 (strided axes only) is the prox along the axis.
template <int MODE>
void run_axis(float2* data, int64_t batch, const int64_t* D, int ax, float thresh, hipStream_t s)
{
    const int N = (int)D[ax];
    const float* fwd = MODE != 1 ? dct_tiles(N, 0, s) : nullptr;
    const float* inv = MODE != 0 ? dct_tiles(N, 1, s) : nullptr;
    const int rt = ((N + 1) / 2 + 15) / 16, pw = (rt + 3) / 4;
    if (ax == 2) {
        if constexpr (MODE != 2) {
            const int64_t nlines = batch * D[0] * D[1], blocks = ceil_div(nlines, kDctCols);
            HASTY_REQUIRE(blocks <= max_blocks(kDctThreads), "too many DCT lines for one launch");
            const size_t smem = sizeof(float) * 2 * kDctCols * line_stride(16 * rt);
            auto kern = pw == 1   ? dct_lines_kernel<1, MODE>
                        : pw == 2 ? dct_lines_kernel<2, MODE>
                        : pw == 3 ? dct_lines_kernel<3, MODE>
                                  : dct_lines_kernel<4, MODE>;
            allow_lds(kern, smem);
            hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kDctThreads), smem, s, data, MODE == 0 ? fwd : inv, N,
                               nlines);
            check_launch("dct_lines_kernel");
        }
        return;
    }
    const int64_t inner = ax == 1 ? D[2] : D[1] * D[2], outer = inner * N;
    const int64_t columns = (ax == 1 ? batch * D[0] : batch) * inner, blocks = ceil_div(columns, kDctCols);
    HASTY_REQUIRE(blocks <= max_blocks(kDctThreads), "too many DCT lines for one launch");
    const size_t smem = sizeof(float) * 2 * 16 * rt * kColStride;
    auto kern = pw == 1   ? dct_strided_kernel<1, MODE>
                : pw == 2 ? dct_strided_kernel<2, MODE>
                : pw == 3 ? dct_strided_kernel<3, MODE>
                          : dct_strided_kernel<4, MODE>;
    allow_lds(kern, smem);
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kDctThreads), smem, s, data, fwd, inv, N, inner, outer, columns,
                       thresh);
    check_launch("dct_strided_kernel");
}

// Axes of the mask longer than 1, with the checks every call makes.
int active_axes(int64_t batch, const int64_t* dims, int axis_mask)
{
    HASTY_REQUIRE(batch >= 0, "batch must be >= 0");
    int m = 0;
    for (int d = 0; d < 3; ++d) {
        HASTY_REQUIRE(dims[d] >= 1, "dims must be >= 1");
        if ((axis_mask & (1 << d)) && dims[d] > 1) m |= 1 << d;
    }
    if (batch > 0)
        for (int d = 0; d < 3; ++d) HASTY_REQUIRE(!(m & (1 << d)) || dims[d] <= 512, "DCT axis longer than 512");
    return m;
}

}  // namespace

void dct3(float2* data, int64_t batch, const int64_t* dims, int axis_mask, int inverse, hipStream_t s)
{
    const int m = active_axes(batch, dims, axis_mask);
    if (batch == 0) return;
    for (int ax = 0; ax < 3; ++ax) {
        if (!(m & (1 << ax))) continue;
        if (inverse) run_axis<1>(data, batch, dims, ax, 0.f, s);
        else run_axis<0>(data, batch, dims, ax, 0.f, s);
    }
}

void l1dct_prox(float2* data, int64_t batch, const int64_t* dims, int axis_mask, float thresh, hipStream_t s)
{
    const int m = active_axes(batch, dims, axis_mask);
    const int64_t n = batch * dims[0] * dims[1] * dims[2];
    if (n == 0) return;
    // the axis whose two transforms run in one pass with the threshold (strided axes only)
    const int mid = (m & 1) ? 0 : (m & 2) ? 1 : -1;
    for (int ax = 2; ax > mid; --ax)
        if (m & (1 << ax)) run_axis<0>(data, batch, dims, ax, 0.f, s);
    if (mid >= 0) {
        run_axis<2>(data, batch, dims, mid, thresh, s);
    } else {
        hipLaunchKernelGGL(soft_kernel, dim3((unsigned)ceil_div(n, kDctThreads)), dim3(kDctThreads), 0, s, data, n,
                           thresh);
        check_launch("soft_kernel");
    }
    for (int ax = mid + 1; ax < 3; ++ax)
        if (m & (1 << ax)) run_axis<1>(data, batch, dims, ax, 0.f, s);
}

}  // namespace hasty_hip
