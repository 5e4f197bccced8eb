// extern "C" entry points of libhasty_hip.so (declared in include/hasty_hip.h) and the
// host-side drivers behind them (LLR block grid, workspace layout).
#include <atomic>
#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>
#include <random>
#include <tuple>
#include <string>
#include <vector>

#include "../../../include/hasty_hip.h"
#include "common.hpp"
#include "fft.hpp"
#include "nufft.hpp"
#include "toeplitz.hpp"
#include "cg.hpp"
#include "llr.hpp"
#include "tune.hpp"

namespace hasty_hip {

namespace {
thread_local std::string g_last_error;
std::atomic<int> g_opt_sense_fused{1};

template <typename Fn> int guarded(Fn&& fn)
{
    try {
        fn();
        return kOk;
    } catch (const HastyError& e) {
        set_last_error(e.what());
        return e.code;
    } catch (const std::bad_alloc&) {
        set_last_error("host out of memory");
        return kOutOfMemory;
    } catch (const std::exception& e) {
        set_last_error(e.what());
        return kHipError;
    } catch (...) {
        set_last_error("unknown error");
        return kHipError;
    }
}

hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// Enumerate the strided block grid of one pass (svt.cpp:393-436), skip rule included.
std::vector<int32_t> grid_blocks(const int64_t* dims5, const int64_t* strides, const int64_t* shape, int sx_, int sy_,
                                 int sz_)
{
    const int64_t Sx = dims5[2], Sy = dims5[3], Sz = dims5[4];
    const int64_t bx = Sx / strides[0], by = Sy / strides[1], bz = Sz / strides[2];
    std::vector<int32_t> out;
    for (int64_t nx = 0; nx < bx; ++nx) {
        const int64_t sx = nx * strides[0] + sx_;
        if (sx + shape[0] >= Sx) continue;
        for (int64_t ny = 0; ny < by; ++ny) {
            const int64_t sy = ny * strides[1] + sy_;
            if (sy + shape[1] >= Sy) continue;
            for (int64_t nz = 0; nz < bz; ++nz) {
                const int64_t sz = nz * strides[2] + sz_;
                if (sz + shape[2] >= Sz) continue;
                out.push_back((int32_t)sx);
                out.push_back((int32_t)sy);
                out.push_back((int32_t)sz);
            }
        }
    }
    return out;
}

// Row splits of the LLR Gram per (blocks per launch, rows, columns), set by
// hasty_autotune_llr; other shapes use the rule in choose_nsplit.
std::map<std::tuple<int64_t, int64_t, int64_t>, int> g_nsplit_tuned;
std::mutex g_nsplit_mu;

int max_nsplit(int64_t R) { return (int)std::min<int64_t>(8, std::max<int64_t>(1, R / 256)); }

int choose_nsplit(int64_t nblk, int64_t R, int64_t F)
{
    {
        std::lock_guard<std::mutex> lock(g_nsplit_mu);
        auto it = g_nsplit_tuned.find(std::make_tuple(nblk, R, F));
        if (it != g_nsplit_tuned.end()) return it->second;
    }
    int64_t ns = ceil_div(512, std::max<int64_t>(1, nblk));
    ns = std::min<int64_t>(ns, max_nsplit(R));
    return (int)std::max<int64_t>(1, ns);
}

size_t llr_ws_bytes_for(int64_t nblk, int64_t F, int64_t R)
{
    const int ns = choose_nsplit(nblk, R, F);
    return 256 + sizeof(int32_t) * 3 * (size_t)nblk + llr_workspace_bytes(nblk, F, ns);
}

// Largest workspace any batch of 1..nmax blocks needs (the split count depends on it).
size_t llr_ws_bound(int64_t nmax, int64_t F, int64_t R)
{
    size_t m = 0;
    for (int64_t n = 1; n <= nmax; ++n) m = std::max(m, llr_ws_bytes_for(n, F, R));
    return m;
}

// Run one batch of disjoint blocks. The corner list is copied into the head of ws.
void run_llr_batch(float2* data, const LlrGeom& g, const std::vector<int32_t>& corners, float thresh, int soft,
                   void* ws, size_t ws_bytes, hipStream_t s)
{
    const int64_t nblk = (int64_t)corners.size() / 3;
    if (nblk == 0) return;
    const int64_t R = g.E * g.bx * g.by * g.bz;
    const int nsplit = choose_nsplit(nblk, R, g.F);
    const size_t cbytes = ((sizeof(int32_t) * 3 * (size_t)nblk + 255) / 256) * 256;
    HASTY_REQUIRE(ws_bytes >= cbytes + llr_workspace_bytes(nblk, g.F, nsplit), "LLR workspace too small");
    int3* cdev = reinterpret_cast<int3*>(ws);
    HASTY_HIP_CHECK(hipMemcpyAsync(cdev, corners.data(), sizeof(int32_t) * corners.size(), hipMemcpyHostToDevice, s));
    const int rank = soft ? 0 : (int)(thresh + 0.5);
    llr_blocks(data, g, cdev, nblk, thresh, soft, rank, static_cast<char*>(ws) + cbytes, ws_bytes - cbytes, nsplit,
               nullptr, s);
    // The host corner list must outlive the async copy.
    HASTY_HIP_CHECK(hipStreamSynchronize(s));
}

LlrGeom image_geom(const int64_t* dims5, const int64_t* shape)
{
    LlrGeom g;
    g.F = dims5[0];
    g.E = dims5[1];
    g.X = dims5[2];
    g.Y = dims5[3];
    g.Z = dims5[4];
    g.bx = (int)shape[0];
    g.by = (int)shape[1];
    g.bz = (int)shape[2];
    g.fstride = g.E * g.X * g.Y * g.Z;
    g.rstride = 1;
    return g;
}

void check_dims5(const int64_t* dims5, const int64_t* shape)
{
    for (int i = 0; i < 5; ++i) HASTY_REQUIRE(dims5[i] >= 1, "image dims must be >= 1");
    for (int i = 0; i < 3; ++i) {
        HASTY_REQUIRE(shape[i] >= 1 && shape[i] <= dims5[2 + i], "block shape must fit the image");
    }
    llr_check(dims5[0]);
}

// Scratch of hasty_svt_matrix_noalloc: the corner of its one block (first 256 B), then
// the Gram partial sums, W and the recorded Jacobi rotations of a block of up to 128
// columns (3.13 MB at 128 columns and 8 row splits). One copy per GPU, alive until the
// process ends; host code reaches it only through the address hipGetSymbolAddress
// returns for the current device (the symbol itself is a host-side stand-in).
constexpr size_t kSvtScratchBytes = size_t(4) << 20;
__device__ __align__(256) unsigned char scratch[kSvtScratchBytes];

std::mutex g_scratch_mu;
std::map<int, void*> g_scratch_ptr;  // device ordinal -> device address of `scratch`

// Address of `scratch` on the current device (looked up once per device).
void* scratch_address()
{
    const int dev = current_device();
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    auto it = g_scratch_ptr.find(dev);
    if (it != g_scratch_ptr.end()) return it->second;
    void* p = nullptr;
    HASTY_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    HASTY_REQUIRE(p != nullptr, "no device address for the static scratch");
    g_scratch_ptr[dev] = p;
    return p;
}

__global__ void zero_corner_kernel(int3* c)
{
    if (threadIdx.x == 0) *c = make_int3(0, 0, 0);
}

}  // namespace

void set_last_error(const std::string& msg) { g_last_error = msg; }

namespace {
thread_local DeviceArena* t_arena = nullptr;
}

DeviceArena::DeviceArena(void* base, size_t bytes) : base_(static_cast<char*>(base)), size_(base ? bytes : 0), outer_(t_arena)
{
    const size_t skew = (256 - reinterpret_cast<uintptr_t>(base) % 256) % 256;
    used_ = std::min(size_, skew);
    t_arena = this;
}

DeviceArena::~DeviceArena() { t_arena = outer_; }

void* DeviceArena::take(size_t bytes)
{
    const size_t need = (bytes + 255) / 256 * 256;
    if (need > size_ - used_) return nullptr;
    void* p = base_ + used_;
    used_ += need;
    return p;
}

void* dev_alloc_table(size_t bytes)
{
    void* p = nullptr;
    if (bytes == 0) bytes = 16;
    HASTY_HIP_CHECK(hipMalloc(&p, bytes));
    return p;
}

void* dev_alloc(size_t bytes)
{
    if (t_arena)
        if (void* p = t_arena->take(std::max<size_t>(bytes, 16))) return p;
    return dev_alloc_table(bytes);
}

void dev_free(void* p)
{
    if (p && !(t_arena && t_arena->owns(p))) (void)hipFree(p);
}

int current_device()
{
    int d = 0;
    HASTY_HIP_CHECK(hipGetDevice(&d));
    return d;
}

}  // namespace hasty_hip

using namespace hasty_hip;

struct hasty_nufft_plan_s {
    NufftPlan* impl;
};

struct hasty_graph_s {
    hipGraph_t graph;
    hipGraphExec_t exec;
    int64_t nodes;
};

extern "C" {

const char* hasty_last_error(void) { return g_last_error.c_str(); }

int hasty_version(void) { return 100; }

int hasty_nufft_makeplan(int type, int dim, const int64_t* nmodes, int iflag, int ntransf, double tol, int fp64,
                         hasty_nufft_plan* plan)
{
    return guarded([&] {
        HASTY_REQUIRE(plan != nullptr && nmodes != nullptr, "null argument");
        *plan = nullptr;
        NufftPlan* p = nufft_makeplan(type, dim, nmodes, iflag, ntransf, tol, fp64);
        *plan = new hasty_nufft_plan_s{p};
    });
}

int hasty_nufft_setpts(hasty_nufft_plan plan, int64_t M, const void* x, const void* y, const void* z, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(plan != nullptr, "null plan");
        nufft_setpts(plan->impl, M, x, y, z, as_stream(stream));
    });
}

int hasty_nufft_execute(hasty_nufft_plan plan, void* c, void* f, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(plan != nullptr, "null plan");
        nufft_execute(plan->impl, c, f, as_stream(stream));
    });
}

int hasty_nufft_set_scale(hasty_nufft_plan plan, double scale)
{
    return guarded([&] {
        HASTY_REQUIRE(plan != nullptr, "null plan");
        plan->impl->scale = scale;
    });
}

int hasty_nufft_destroy(hasty_nufft_plan plan)
{
    return guarded([&] {
        if (!plan) return;
        nufft_destroy(plan->impl);
        delete plan;
    });
}

int hasty_nufft_info(hasty_nufft_plan plan, int64_t* nf, int* ns, double* beta)
{
    return guarded([&] {
        HASTY_REQUIRE(plan != nullptr, "null plan");
        const NufftPlan* p = plan->impl;
        for (int d = 0; d < p->dim; ++d)
            if (nf) nf[d] = p->nf[2 - d];
        if (ns) *ns = p->ns;
        if (beta) *beta = p->beta;
    });
}

int hasty_toeplitz_build(const void* coords, int coord_fp64, int64_t M, int ndim, const int64_t* nmodes,
                         const float* weights, void* diag_ref, float* kernel, double tol, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(coords != nullptr || M == 0, "null coords");
        HASTY_REQUIRE(nmodes != nullptr, "null nmodes");
        toeplitz_build(coords, coord_fp64, M, ndim, nmodes, weights, reinterpret_cast<float2*>(diag_ref), kernel, tol,
                       as_stream(stream));
    });
}

size_t hasty_toeplitz_workspace_size(int64_t M, int ndim, const int64_t* nmodes, double tol)
{
    if (M < 0 || ndim < 1 || ndim > 3 || !nmodes || !(tol > 0.0)) return 0;
    return toeplitz_workspace_bytes(M, ndim, nmodes, tol);
}

int hasty_toeplitz_build_ws(const void* coords, int coord_fp64, int64_t M, int ndim, const int64_t* nmodes,
                            const float* weights, void* diag_ref, float* kernel, double tol, void* workspace,
                            size_t workspace_bytes, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(coords != nullptr || M == 0, "null coords");
        HASTY_REQUIRE(nmodes != nullptr, "null nmodes");
        HASTY_REQUIRE(workspace != nullptr || workspace_bytes == 0, "null workspace");
        toeplitz_build(coords, coord_fp64, M, ndim, nmodes, weights, reinterpret_cast<float2*>(diag_ref), kernel, tol,
                       as_stream(stream), workspace, workspace_bytes);
    });
}

int hasty_toeplitz_apply(const void* in, void* out, const void* mul, const void* diag, int ntransf, int ndim,
                         const int64_t* nmodes, int mode, void* storage1, void* storage2, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(in && out && diag && storage1 && storage2 && nmodes, "null argument");
        toeplitz_apply_ref((const float2*)in, (float2*)out, (const float2*)mul, (const float2*)diag, ntransf, ndim, nmodes,
                           mode, (float2*)storage1, (float2*)storage2, as_stream(stream));
    });
}

size_t hasty_sense_normal_workspace_size(const int64_t* nmodes3, int coil_batch, int problem_batch)
{
    if (!nmodes3 || coil_batch < 1) return 0;
    return sense_normal_workspace_bytes(nmodes3, coil_batch, problem_batch);
}

int hasty_sense_normal_prepare(const float* natural, float* prepared, int64_t nk, const int64_t* nmodes3, int* layout,
                               void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(natural && prepared && nmodes3 && layout, "null argument");
        for (int d = 0; d < 3; ++d) HASTY_REQUIRE(nmodes3[d] >= 1, "nmodes must be >= 1");
        const int l = sense_kernel_layout(nmodes3, g_opt_sense_fused != 0);
        HASTY_REQUIRE(l == 0 || prepared != natural, "the fused layout cannot be prepared in place");
        sense_prepare_kernels(natural, prepared, nk, nmodes3, l, as_stream(stream));
        *layout = l;
    });
}

int hasty_sense_normal_toeplitz_ex(const void* x, void* out, const void* smaps, int64_t nsmaps, const int32_t* coils,
                                   int ncoil, int coil_problem_stride, const int32_t* problem_ncoil_host,
                                   const int32_t* problem_ncoil_dev, const float* kernels, int nkernels, int layout,
                                   const int32_t* kernel_index, const void* sub, int nproblems,
                                   const int64_t* nmodes3, void* workspace, size_t workspace_bytes, int coil_batch,
                                   void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(x && out && smaps && coils && kernels && kernel_index && nmodes3 && workspace, "null argument");
        HASTY_REQUIRE(nproblems >= 1, "nproblems must be >= 1");
        HASTY_REQUIRE(coil_problem_stride >= 0, "coil_problem_stride must be >= 0");
        HASTY_REQUIRE(nsmaps < 0 || (int64_t)(nproblems - 1) * coil_problem_stride < nsmaps,
                      "coil_problem_stride reaches past the coil maps");
        HASTY_REQUIRE(!problem_ncoil_dev || problem_ncoil_host, "give the host copy of the per-problem coil counts");
        for (int p = 0; p < nproblems; ++p)
            HASTY_REQUIRE(kernel_index[p] >= 0 && kernel_index[p] < nkernels, "kernel index out of range");
        for (int d = 0; d < 3; ++d) HASTY_REQUIRE(nmodes3[d] >= 1, "nmodes must be >= 1");
        sense_normal_toeplitz((const float2*)x, (float2*)out, (const float2*)smaps, coils, ncoil, kernels, layout,
                              kernel_index, (const float2*)sub, nproblems, nmodes3, workspace, workspace_bytes,
                              coil_batch, as_stream(stream), coil_problem_stride, problem_ncoil_host,
                              problem_ncoil_dev);
    });
}

int hasty_sense_normal_toeplitz(const void* x, void* out, const void* smaps, const int32_t* coils, int ncoil,
                                const float* kernels, int nkernels, int layout, const int32_t* kernel_index,
                                const void* sub, int nproblems, const int64_t* nmodes3, void* workspace,
                                size_t workspace_bytes, int coil_batch, void* stream)
{
    return hasty_sense_normal_toeplitz_ex(x, out, smaps, -1, coils, ncoil, 0, nullptr, nullptr, kernels, nkernels,
                                          layout, kernel_index, sub, nproblems, nmodes3, workspace, workspace_bytes,
                                          coil_batch, stream);
}

int hasty_set_option(const char* name, int64_t value)
{
    if (name && std::strcmp(name, "sense_fused") == 0) {
        g_opt_sense_fused = (int)value;
        return 0;
    }
    if (name && std::strcmp(name, "sense_xy_variant") == 0 && value >= 0 && value <= 3) {
        sense_fused_set_xy_variant((int)value);
        return 0;
    }
    if (name && std::strcmp(name, "nufft_spread_variant") == 0 && value >= 0 && value <= 6) {
        nufft_set_spread_variant((int)value);
        return 0;
    }
    if (name && std::strcmp(name, "sense_zconv_batch") == 0 && value >= 1 && value <= 16) {
        sense_fused_set_zconv_batch((int)value);
        return 0;
    }
    if (name && std::strcmp(name, "llr_eig_threads") == 0 && (value == 256 || value == 512 || value == 768)) {
        llr_set_eig_threads((int)value);
        return 0;
    }
    if (name && std::strcmp(name, "llr_max_sweeps") == 0 && value >= 1 && value <= 15) {
        llr_set_max_sweeps((int)value);
        return 0;
    }
    if (name && std::strcmp(name, "sense_zconv_variant") == 0 && value >= 0 && value <= 3) {
        sense_fused_set_zconv_variant((int)value);
        return 0;
    }
    if (name && std::strcmp(name, "nufft_locality") == 0 && value >= 0 && value <= 4) {
        nufft_set_locality((int)value);
        return 0;
    }
    if (name && std::strcmp(name, "nufft_spread_tile") == 0 && (value == 0 || (value >= 12 && value <= 28))) {
        nufft_set_tile((int)value);
        return 0;
    }
    if (name && std::strcmp(name, "nufft_spread_chunk") == 0 && (value == 0 || (value >= 32 && value <= 8192))) {
        nufft_set_chunk((int)value);
        return 0;
    }
    if (name && std::strcmp(name, "fft_r16") == 0 && (value == 0 || value == 1)) {
        fft_set_r16((int)value);
        return 0;
    }
    if (name && std::strcmp(name, "fft_strided_lines") == 0 && value >= 0 && value <= 64) {
        fft_set_strided_lines((int)value);
        return 0;
    }
    set_last_error(std::string("unknown option ") + (name ? name : "(null)"));
    return 1;
}

int hasty_get_option(const char* name, int64_t* value)
{
    if (!value) {
        set_last_error("value must not be NULL");
        return 1;
    }
    if (name && std::strcmp(name, "sense_fused") == 0) *value = g_opt_sense_fused;
    else if (name && std::strcmp(name, "sense_xy_variant") == 0) *value = sense_fused_get_xy_variant();
    else if (name && std::strcmp(name, "nufft_spread_variant") == 0) *value = nufft_get_spread_variant();
    else if (name && std::strcmp(name, "sense_zconv_batch") == 0) *value = sense_fused_get_zconv_batch();
    else if (name && std::strcmp(name, "llr_max_sweeps") == 0) *value = llr_get_max_sweeps();
    else if (name && std::strcmp(name, "llr_eig_threads") == 0) *value = llr_get_eig_threads();
    else if (name && std::strcmp(name, "sense_zconv_variant") == 0) *value = sense_fused_get_zconv_variant();
    else if (name && std::strcmp(name, "nufft_spread_tile") == 0) *value = nufft_get_tile();
    else if (name && std::strcmp(name, "nufft_spread_chunk") == 0) *value = nufft_get_chunk();
    else if (name && std::strcmp(name, "nufft_locality") == 0) *value = nufft_get_locality();
    else if (name && std::strcmp(name, "fft_strided_lines") == 0) *value = fft_get_strided_lines();
    else if (name && std::strcmp(name, "fft_r16") == 0) *value = fft_get_r16();
    else {
        set_last_error(std::string("unknown option ") + (name ? name : "(null)"));
        return 1;
    }
    return 0;
}

int hasty_timing_enable(int on)
{
    return guarded([&] { timing_enable(on != 0); });
}

int hasty_timing_entries(void)
{
    int n = -1;
    if (guarded([&] { n = timing_entries(); }) != 0) return -1;
    return n;
}

int hasty_timing_read(int index, char* name, int name_capacity, double* total_ms, int64_t* count)
{
    return guarded([&] {
        HASTY_REQUIRE(name && name_capacity > 0 && total_ms && count, "null argument");
        std::string nm;
        HASTY_REQUIRE(timing_read(index, &nm, total_ms, count), "timing index out of range");
        const size_t n = std::min(nm.size(), (size_t)name_capacity - 1);
        std::memcpy(name, nm.data(), n);
        name[n] = '\0';
    });
}

size_t hasty_cg_workspace_size(int64_t nproblems, int64_t n)
{
    return sizeof(double) * cg_workspace_doubles(nproblems, n);
}

int hasty_cg_init(int64_t nproblems, int64_t n, const void* b, const void* Ax, void* r, void* p, double* state,
                  void* workspace, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(b && Ax && r && p && state && workspace, "null argument");
        cg_init(nproblems, n, (const float2*)b, (const float2*)Ax, (float2*)r, (float2*)p, state, (double*)workspace,
                as_stream(stream));
    });
}

int hasty_cg_iterate(int64_t nproblems, int64_t n, void* x, void* r, void* p, const void* Ap, double* state,
                     void* workspace, double tol, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(x && r && p && Ap && state && workspace, "null argument");
        cg_iterate(nproblems, n, (float2*)x, (float2*)r, (float2*)p, (const float2*)Ap, state, (double*)workspace, tol,
                   as_stream(stream));
    });
}

int hasty_cg_iterate_l2(int64_t nproblems, int64_t n, void* x, void* r, void* p, const void* Ap, double* state,
                        void* workspace, double tol, double lambda, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(x && r && p && Ap && state && workspace, "null argument");
        cg_iterate(nproblems, n, (float2*)x, (float2*)r, (float2*)p, (const float2*)Ap, state, (double*)workspace, tol,
                   as_stream(stream), lambda);
    });
}

int hasty_cg_init_precond(int64_t nproblems, int64_t n, const void* r, const void* z, void* p, double* state,
                          void* workspace, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(r && z && p && state && workspace, "null argument");
        cg_init_precond(nproblems, n, (const float2*)r, (const float2*)z, (float2*)p, state, (double*)workspace,
                        as_stream(stream));
    });
}

int hasty_cg_iterate_xr(int64_t nproblems, int64_t n, void* x, void* r, const void* p, const void* Ap, double* state,
                        void* workspace, double tol, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(x && r && p && Ap && state && workspace, "null argument");
        cg_iterate_xr(nproblems, n, (float2*)x, (float2*)r, (const float2*)p, (const float2*)Ap, state,
                      (double*)workspace, tol, as_stream(stream));
    });
}

int hasty_cg_iterate_pz(int64_t nproblems, int64_t n, const void* r, const void* z, void* p, double* state,
                        void* workspace, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(r && z && p && state && workspace, "null argument");
        cg_iterate_pz(nproblems, n, (const float2*)r, (const float2*)z, (float2*)p, state, (double*)workspace,
                      as_stream(stream));
    });
}

int hasty_circulant_precond_build(const void* smaps, int64_t ncoil, const void* coords, int coord_fp64, int64_t M,
                                  int ndim, const int64_t* nmodes, const float* weights, double lambda, int centered,
                                  void* diag, double tol, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(smaps && nmodes && diag && (coords || M == 0), "null argument");
        circulant_precond_build((const float2*)smaps, ncoil, coords, coord_fp64, M, ndim, nmodes, weights, lambda,
                                centered, (float2*)diag, tol, as_stream(stream));
    });
}

size_t hasty_circulant_precond_workspace_size(int64_t ndiag, int ndim, const int64_t* nmodes, int centered, int adjoint)
{
    if (!nmodes || ndim < 1 || ndim > 3) return 0;
    return circulant_precond_workspace_bytes(ndiag, ndim, nmodes, centered, adjoint);
}

int hasty_circulant_precond_apply(const void* in, void* out, const void* diag, int64_t ndiag, int64_t nproblems,
                                  const int32_t* diag_index, int ndim, const int64_t* nmodes, int centered,
                                  int adjoint, void* workspace, size_t workspace_bytes, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(in && out && diag && nmodes, "null argument");
        circulant_precond_apply((const float2*)in, (float2*)out, (const float2*)diag, ndiag, nproblems, diag_index,
                                ndim, nmodes, centered, adjoint, workspace, workspace_bytes, as_stream(stream));
    });
}

int hasty_dct3(void* data, int64_t batch, const int64_t* dims3, int axis_mask, int inverse, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(data && dims3, "null argument");
        dct3((float2*)data, batch, dims3, axis_mask, inverse, as_stream(stream));
    });
}

int hasty_l1dct_prox(void* data, int64_t batch, const int64_t* dims3, int axis_mask, double thresh, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(data && dims3, "null argument");
        l1dct_prox((float2*)data, batch, dims3, axis_mask, (float)thresh, as_stream(stream));
    });
}

int hasty_llr_shifts(int64_t block_iter, const int64_t* block_shape, int32_t* shifts)
{
    return guarded([&] {
        HASTY_REQUIRE(block_iter >= 1, "Can't perform Normal3DBlocksSVT with block_iter < 1");
        HASTY_REQUIRE(block_shape && shifts, "null argument");
        std::default_random_engine generator;
        for (int d = 0; d < 3; ++d) {
            shifts[d * block_iter] = 0;
            if (block_iter > 1) {
                std::uniform_int_distribution<int> distribution(0, (int)block_shape[d]);
                for (int64_t b = 1; b < block_iter; ++b) shifts[d * block_iter + b] = distribution(generator);
            }
        }
    });
}

size_t hasty_llr_workspace_size(const int64_t* dims5, const int64_t* block_strides, const int64_t* block_shape)
{
    if (!dims5 || !block_strides || !block_shape) return 0;
    int64_t nmax = 1;
    for (int d = 0; d < 3; ++d) {
        if (block_strides[d] < 1) return 0;
        nmax *= std::max<int64_t>(1, dims5[2 + d] / block_strides[d]);
    }
    const int64_t R = dims5[1] * block_shape[0] * block_shape[1] * block_shape[2];
    return llr_ws_bound(nmax, dims5[0], R);
}

int hasty_llr_normal_blocks(void* data, const int64_t* dims5, const int64_t* block_strides,
                            const int64_t* block_shape, int64_t block_iter, const int32_t* shifts, double thresh,
                            int soft, void* workspace, size_t workspace_bytes, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(data && dims5 && block_strides && block_shape && workspace, "null argument");
        HASTY_REQUIRE(block_iter >= 1, "Can't perform Normal3DBlocksSVT with block_iter < 1");
        HASTY_REQUIRE(thresh >= 0.0, "threshold must be >= 0");
        for (int d = 0; d < 3; ++d) HASTY_REQUIRE(block_strides[d] >= 1, "block strides must be >= 1");
        check_dims5(dims5, block_shape);
        std::vector<int32_t> sh(3 * block_iter);
        if (shifts) {
            std::memcpy(sh.data(), shifts, sizeof(int32_t) * sh.size());
        } else {
            if (hasty_llr_shifts(block_iter, block_shape, sh.data())) throw HastyError(kInvalidArgument, g_last_error);
        }
        const LlrGeom g = image_geom(dims5, block_shape);
        const bool disjoint = block_strides[0] >= block_shape[0] && block_strides[1] >= block_shape[1] &&
                              block_strides[2] >= block_shape[2];
        hipStream_t s = as_stream(stream);
        for (int64_t it = 0; it < block_iter; ++it) {
            std::vector<int32_t> blocks = grid_blocks(dims5, block_strides, block_shape, sh[0 * block_iter + it],
                                                      sh[1 * block_iter + it], sh[2 * block_iter + it]);
            if (disjoint) {
                run_llr_batch((float2*)data, g, blocks, (float)thresh, soft, workspace, workspace_bytes, s);
            } else {
                // Overlapping blocks within a pass: keep the reference's sequential order.
                for (size_t b = 0; b < blocks.size(); b += 3) {
                    std::vector<int32_t> one(blocks.begin() + b, blocks.begin() + b + 3);
                    run_llr_batch((float2*)data, g, one, (float)thresh, soft, workspace, workspace_bytes, s);
                }
            }
        }
    });
}

int hasty_llr_blocks(void* data, const int64_t* dims5, const int64_t* block_shape, const int32_t* corners,
                     int64_t nblk, double thresh, int soft, void* workspace, size_t workspace_bytes, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(data && dims5 && block_shape && workspace, "null argument");
        HASTY_REQUIRE(nblk >= 0 && (nblk == 0 || corners), "null corners");
        HASTY_REQUIRE(thresh >= 0.0, "threshold must be >= 0");
        check_dims5(dims5, block_shape);
        for (int64_t b = 0; b < nblk; ++b)
            for (int d = 0; d < 3; ++d)
                HASTY_REQUIRE(corners[3 * b + d] >= 0 && corners[3 * b + d] + block_shape[d] <= dims5[2 + d],
                              "block outside the image");
        std::vector<int32_t> c(corners, corners + 3 * nblk);
        run_llr_batch((float2*)data, image_geom(dims5, block_shape), c, (float)thresh, soft, workspace,
                      workspace_bytes, as_stream(stream));
    });
}

int hasty_llr_grid_corners(const int64_t* dims5, const int64_t* block_strides, const int64_t* block_shape,
                           const int32_t* shift3, int32_t* corners_out, int64_t capacity, int64_t* count)
{
    return guarded([&] {
        HASTY_REQUIRE(dims5 && block_strides && block_shape && shift3 && count, "null argument");
        for (int d = 0; d < 3; ++d) HASTY_REQUIRE(block_strides[d] >= 1, "block strides must be >= 1");
        check_dims5(dims5, block_shape);
        const std::vector<int32_t> b = grid_blocks(dims5, block_strides, block_shape, shift3[0], shift3[1], shift3[2]);
        *count = (int64_t)b.size() / 3;
        HASTY_REQUIRE(!corners_out || capacity >= *count, "corner buffer too small");
        if (corners_out) std::memcpy(corners_out, b.data(), sizeof(int32_t) * b.size());
    });
}

int hasty_llr_blocks_dev(void* data, const int64_t* dims5, const int64_t* block_shape, const int32_t* corners_dev,
                         int64_t nblk, double thresh, int soft, void* workspace, size_t workspace_bytes, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(data && dims5 && block_shape && workspace, "null argument");
        HASTY_REQUIRE(nblk >= 0 && (nblk == 0 || corners_dev), "null corners");
        HASTY_REQUIRE(thresh >= 0.0, "threshold must be >= 0");
        check_dims5(dims5, block_shape);
        if (nblk == 0) return;
        const LlrGeom g = image_geom(dims5, block_shape);
        const int nsplit = choose_nsplit(nblk, g.E * g.bx * g.by * g.bz, g.F);
        HASTY_REQUIRE(workspace_bytes >= llr_workspace_bytes(nblk, g.F, nsplit), "LLR workspace too small");
        const int rank = soft ? 0 : (int)(thresh + 0.5);
        llr_blocks((float2*)data, g, reinterpret_cast<const int3*>(corners_dev), nblk, (float)thresh, soft, rank,
                   workspace, workspace_bytes, nsplit, nullptr, as_stream(stream));
    });
}

size_t hasty_svt_workspace_size(int64_t R, int64_t F) { return llr_ws_bound(1, F, R); }

size_t hasty_llr_blocks_workspace_size(const int64_t* dims5, const int64_t* block_shape, int64_t nblk)
{
    if (!dims5 || !block_shape || nblk < 0) return 0;
    const int64_t R = dims5[1] * block_shape[0] * block_shape[1] * block_shape[2];
    return llr_ws_bytes_for(std::max<int64_t>(1, nblk), dims5[0], R);
}

int hasty_svt_matrix(void* A, int64_t R, int64_t F, double thresh, int soft, void* workspace, size_t workspace_bytes,
                     void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(A && workspace, "null argument");
        HASTY_REQUIRE(R >= 1, "matrix must have rows");
        HASTY_REQUIRE(thresh >= 0.0, "threshold must be >= 0");
        llr_check(F);
        // A row-major [R][F] matrix is a one-block "image" F x 1 x 1 x 1 x R whose
        // column stride is 1 and row stride F.
        LlrGeom g;
        g.F = F;
        g.E = 1;
        g.X = 1;
        g.Y = 1;
        g.Z = R;
        g.bx = 1;
        g.by = 1;
        g.bz = (int)R;
        g.fstride = 1;
        g.rstride = F;
        std::vector<int32_t> c = {0, 0, 0};
        run_llr_batch((float2*)A, g, c, (float)thresh, soft, workspace, workspace_bytes, as_stream(stream));
    });
}

int hasty_svt_matrix_noalloc(void* A, int64_t R, int64_t F, double thresh, int soft, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(A, "null argument");
        HASTY_REQUIRE(R >= 1, "matrix must have rows");
        HASTY_REQUIRE(thresh >= 0.0, "threshold must be >= 0");
        llr_check(F);
        // the matrix as a one-block image, as in hasty_svt_matrix
        LlrGeom g;
        g.F = F;
        g.E = 1;
        g.X = 1;
        g.Y = 1;
        g.Z = R;
        g.bx = 1;
        g.by = 1;
        g.bz = (int)R;
        g.fstride = 1;
        g.rstride = F;
        const int nsplit = choose_nsplit(1, R, F);
        const size_t need = 256 + llr_workspace_bytes(1, F, nsplit);
        HASTY_REQUIRE(need <= kSvtScratchBytes, "hasty_svt_matrix_noalloc: the block needs " + std::to_string(need) +
                                                    " bytes of scratch, more than the static " +
                                                    std::to_string(kSvtScratchBytes));
        hipStream_t s = as_stream(stream);
        unsigned char* ws = static_cast<unsigned char*>(scratch_address());
        int3* corner = reinterpret_cast<int3*>(ws);
        hipLaunchKernelGGL(zero_corner_kernel, dim3(1), dim3(64), 0, s, corner);
        check_launch("zero_corner_kernel");
        const int rank = soft ? 0 : (int)(thresh + 0.5);
        llr_blocks((float2*)A, g, corner, 1, (float)thresh, soft, rank, ws + 256, kSvtScratchBytes - 256, nsplit,
                   nullptr, s);
    });
}

int hasty_autotune_sense_normal(const int64_t* nmodes3, int ncoil, int nproblems, int64_t* choice,
                                double* ms_per_problem, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(nmodes3 && choice, "null argument");
        for (int d = 0; d < 3; ++d) HASTY_REQUIRE(nmodes3[d] >= 1, "nmodes must be >= 1");
        const SenseChoice c = autotune_sense_normal(nmodes3, ncoil, nproblems, g_opt_sense_fused != 0,
                                                    as_stream(stream));
        choice[0] = c.xy_variant;
        choice[1] = c.zconv_batch;
        choice[2] = c.problem_batch;
        choice[3] = c.coil_batch;
        choice[4] = c.zconv_variant;
        if (ms_per_problem) *ms_per_problem = c.ms_per_problem;
    });
}

int hasty_nufft_autotune(hasty_nufft_plan plan, void* c, void* f, int64_t* spread_variant, double* ms, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(plan != nullptr, "null plan");
        const int v = nufft_autotune(plan->impl, c, f, as_stream(stream), ms);
        if (spread_variant) *spread_variant = v;
    });
}

int hasty_nufft_plan_shape(hasty_nufft_plan plan, int64_t* tile, int64_t* chunk, int64_t* spread_variant)
{
    return guarded([&] {
        HASTY_REQUIRE(plan != nullptr, "null plan");
        const NufftPlan* p = plan->impl;
        if (tile) *tile = p->dim == 3 ? nufft_tile_edge(p) : 0;
        if (chunk) *chunk = p->chunk;
        if (spread_variant) *spread_variant = p->spread_variant >= 0 ? p->spread_variant : nufft_get_spread_variant();
    });
}

int hasty_autotune_llr(const int64_t* dims5, const int64_t* block_strides, const int64_t* block_shape,
                       int64_t* nsplit, double* ms, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(dims5 && block_strides && block_shape, "null argument");
        for (int d = 0; d < 3; ++d) HASTY_REQUIRE(block_strides[d] >= 1, "block strides must be >= 1");
        check_dims5(dims5, block_shape);
        hipStream_t s = as_stream(stream);
        const LlrGeom g = image_geom(dims5, block_shape);
        const std::vector<int32_t> blocks = grid_blocks(dims5, block_strides, block_shape, 0, 0, 0);
        const int64_t nblk = (int64_t)blocks.size() / 3;
        const int64_t R = g.E * g.bx * g.by * g.bz;
        if (nblk == 0) {
            if (nsplit) *nsplit = 1;
            if (ms) *ms = 0.0;
            return;
        }
        const auto key = std::make_tuple(nblk, R, g.F);
        {
            std::lock_guard<std::mutex> lock(g_nsplit_mu);
            g_nsplit_tuned.erase(key);
        }
        const int ns0 = choose_nsplit(nblk, R, g.F);
        const int64_t nval = dims5[0] * dims5[1] * dims5[2] * dims5[3] * dims5[4];
        void* img = dev_alloc(sizeof(float2) * nval);
        void* ws = nullptr;
        int best = ns0;
        double tbest = 1e300;
        try {
            fill_uniform((float*)img, 2 * nval, 7u, -1.f, 1.f, s);
            std::vector<int> order = {ns0};
            for (int v : {1, 2, 4, 8})
                if (v != ns0 && v <= max_nsplit(R)) order.push_back(v);
            for (int v : order) {
                {
                    std::lock_guard<std::mutex> lock(g_nsplit_mu);
                    g_nsplit_tuned[key] = v;
                }
                const size_t wsb = llr_ws_bytes_for(nblk, g.F, R);
                dev_free(ws);
                ws = nullptr;
                ws = dev_alloc(wsb);
                // threshold 0: W = I, so the data stays as it is between runs
                const double t = time_best_ms(
                    [&] { run_llr_batch((float2*)img, g, blocks, 0.f, 1, ws, wsb, s); }, s, 3);
                if (t < 0.98 * tbest) {
                    tbest = t;
                    best = v;
                }
            }
            // the eigensolver's workgroup size (a process-wide option) with that split
            {
                std::lock_guard<std::mutex> lock(g_nsplit_mu);
                g_nsplit_tuned[key] = best;
            }
            const int nth0 = llr_get_eig_threads();
            int best_nth = nth0;
            // the workspace of the chosen split (the loop above left the last tried one's)
            const size_t wsb = llr_ws_bytes_for(nblk, g.F, R);
            dev_free(ws);
            ws = nullptr;
            ws = dev_alloc(wsb);
            for (int nth : {256, 512, 768}) {
                if (nth == nth0) continue;
                llr_set_eig_threads(nth);
                const double t = time_best_ms(
                    [&] { run_llr_batch((float2*)img, g, blocks, 0.f, 1, ws, wsb, s); }, s, 3);
                if (t < 0.98 * tbest) {
                    tbest = t;
                    best_nth = nth;
                }
            }
            llr_set_eig_threads(best_nth);
        } catch (...) {
            dev_free(ws);
            dev_free(img);
            std::lock_guard<std::mutex> lock(g_nsplit_mu);
            g_nsplit_tuned.erase(key);
            throw;
        }
        dev_free(ws);
        dev_free(img);
        {
            std::lock_guard<std::mutex> lock(g_nsplit_mu);
            g_nsplit_tuned[key] = best;
        }
        if (nsplit) *nsplit = best;
        if (ms) *ms = tbest;
    });
}

int hasty_stream_probe(int nread, int nwrite, int nontemporal, const void* const* src, void* const* dst,
                       int64_t bytes, void* stream)
{
    return guarded([&] { stream_probe(nread, nwrite, nontemporal != 0, src, dst, bytes, as_stream(stream)); });
}

int hasty_graph_begin(void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(stream != nullptr, "the NULL stream cannot be captured; use a created stream");
        HASTY_HIP_CHECK(hipStreamBeginCapture(as_stream(stream), hipStreamCaptureModeThreadLocal));
    });
}

int hasty_graph_end(void* stream, hasty_graph* graph)
{
    return guarded([&] {
        HASTY_REQUIRE(stream != nullptr && graph != nullptr, "null argument");
        *graph = nullptr;
        hipGraph_t g = nullptr;
        HASTY_HIP_CHECK(hipStreamEndCapture(as_stream(stream), &g));
        HASTY_REQUIRE(g != nullptr, "the capture produced no graph");
        size_t nodes = 0;
        hipGraphExec_t e = nullptr;
        hipError_t err = hipGraphGetNodes(g, nullptr, &nodes);
        if (err == hipSuccess) err = hipGraphInstantiate(&e, g, nullptr, nullptr, 0);
        if (err != hipSuccess) {
            (void)hipGraphDestroy(g);
            HASTY_HIP_CHECK(err);
        }
        *graph = new hasty_graph_s{g, e, (int64_t)nodes};
    });
}

int hasty_graph_launch(hasty_graph graph, void* stream)
{
    return guarded([&] {
        HASTY_REQUIRE(graph != nullptr, "null graph");
        HASTY_REQUIRE(stream != nullptr, "graphs launch on a created stream, not the NULL stream");
        HASTY_HIP_CHECK(hipGraphLaunch(graph->exec, as_stream(stream)));
    });
}

int64_t hasty_graph_nodes(hasty_graph graph) { return graph ? graph->nodes : -1; }

int hasty_graph_destroy(hasty_graph graph)
{
    return guarded([&] {
        if (!graph) return;
        hipError_t e1 = graph->exec ? hipGraphExecDestroy(graph->exec) : hipSuccess;
        hipError_t e2 = graph->graph ? hipGraphDestroy(graph->graph) : hipSuccess;
        delete graph;
        HASTY_HIP_CHECK(e1);
        HASTY_HIP_CHECK(e2);
    });
}

}  // extern "C"
