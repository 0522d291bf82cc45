// Kernels compiled ahead of time for gfx950 (everything that depends on the
// user's system is compiled at run time by hipRTC instead).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstring>
#include <mutex>
#include <string>

#include "../../include/sodecl.h"
#include "device/sin.hip"
#include "device/random.hip"
#include "device/gauss.hip"
#include "sodecl_internal.hpp"

// ---------------------------------------------------------------------------
// Static scratch of sodecl_adjoint_device_noalloc: the backward sweep's
// workspace for callers that cannot allocate device memory.  Every GPU the
// library runs on holds its own copy (64 MiB) until the process ends.  Host
// code never passes the array's name to a kernel (on the host it is a
// stand-in, not a device address): the address each device gives for it is
// resolved once per device with hipGetSymbolAddress and used instead.
// ---------------------------------------------------------------------------
#define SODECL_SCRATCH_DOUBLES ((size_t)8 << 20)
#define SODECL_SCRATCH_DEVICES 64

static __device__ __align__(256) double scratch[SODECL_SCRATCH_DOUBLES];

namespace {
std::mutex scratch_mutex;
double* scratch_ptr[SODECL_SCRATCH_DEVICES];
}  // namespace

namespace sodecl_amd {

size_t scratch_doubles() { return SODECL_SCRATCH_DOUBLES; }

double* scratch_address(int device, std::string& err)
{
    if (device < 0 || device >= SODECL_SCRATCH_DEVICES) {
        err = "device ordinal out of range for the scratch table";
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(scratch_mutex);
    hipError_t e = hipSetDevice(device);
    if (e != hipSuccess) {
        err = std::string("hipSetDevice: ") + hipGetErrorString(e);
        return nullptr;
    }
    if (!scratch_ptr[device]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            err = std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
            return nullptr;
        }
        scratch_ptr[device] = (double*)p;
    }
    return scratch_ptr[device];
}

}  // namespace sodecl_amd

extern "C" int sodecl_adjoint_device_noalloc(sodecl_ctx* ctx, const double* ckpt_t, const double* ckpt_y,
                                             const double* params, const double* cot, double* grad_y0,
                                             double* grad_params, int ckpt_every, void* stream)
{
    if (!ctx) return 0;
    std::string err;
    double* work = sodecl_amd::scratch_address(ctx->device, err);
    if (!work) return sodecl_amd::fail(ctx, err);
    return sodecl_amd::adjoint_into_workspace(ctx, ckpt_t, ckpt_y, params, cot, grad_y0, grad_params, work,
                                              SODECL_SCRATCH_DOUBLES, ckpt_every, stream);
}

// Plain streaming copy, 16 bytes per lane per iteration, grid-stride: the
// reference point for reading HBM traffic counters (bytes fetched and written
// by a kernel of known size).
__global__ void __launch_bounds__(256) sodecl_calibration_copy(const double2* __restrict__ src,
                                                                double2* __restrict__ dst, size_t n)
{
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

extern "C" int sodecl_copy_device(void* dst, const void* src, size_t bytes, void* stream)
{
    if (!dst || !src || bytes % 16 != 0) return 0;
    const size_t n = bytes / 16;
    if (n == 0) return 1;
    int device = 0;
    (void)hipGetDevice(&device);
    int cus = 256;
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
    size_t blocks = (n + 255) / 256;
    const size_t cap = (size_t)cus * 8;
    if (blocks > cap) blocks = cap;
    hipLaunchKernelGGL(sodecl_calibration_copy, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                       (const double2*)src, (double2*)dst, n);
    return hipGetLastError() == hipSuccess ? 1 : 0;
}

// Diagnostic: Threefry-2x64-20 blocks and their open-interval doubles,
// computed by the same device functions the integrators and the sampler
// compile.  in[i] = {ctr0, ctr1, key0, key1}; out[i] = {word0, word1, bits of
// u01(word0), bits of u01(word1)}.
__global__ void __launch_bounds__(256) sodecl_threefry_blocks(const sodecl_u64* __restrict__ in,
                                                               sodecl_u64* __restrict__ out, size_t n)
{
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        sodecl_u64 w0, w1;
        sodecl_threefry2x64_20(in[4 * i], in[4 * i + 1], in[4 * i + 2], in[4 * i + 3], &w0, &w1);
        out[4 * i] = w0;
        out[4 * i + 1] = w1;
        out[4 * i + 2] = (sodecl_u64)__double_as_longlong(sodecl_u01(w0));
        out[4 * i + 3] = (sodecl_u64)__double_as_longlong(sodecl_u01(w1));
    }
}

extern "C" int sodecl_threefry_device(const uint64_t* in, uint64_t* out, size_t n, void* stream)
{
    if (!in || !out) return 0;
    if (n == 0) return 1;
    size_t blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(sodecl_threefry_blocks, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                       (const sodecl_u64*)in, (sodecl_u64*)out, n);
    return hipGetLastError() == hipSuccess ? 1 : 0;
}

// Draws of sodecl_sample_device: entry (row, col) of out[rows][cols] comes
// from one Threefry-2x64-20 block with counter {row, col} and key
// {seed, SODECL_SAMPLE_KEY1}, so every entry is reproducible on its own
// whatever the launch shape.  u0, u1 = open-open (0, 1) doubles of the two
// output words.  The distributions of up to 120 columns travel by value in
// the kernel arguments (no device allocation; wider tables take several
// launches).
//
// Bound by VALU issue: 110 instructions of Threefry per entry and 30 to 120 of
// the distribution's functions against 8 bytes written.  With consecutive
// entries of a row on consecutive lanes, a wavefront of a mixed table ran
// every distribution's code for each of its entries (526 instructions per
// entry, 262144 x 65 entries in 251 us).  Here a wavefront draws 64 rows of one
// column, whose distribution is then the same for all its lanes, and a block
// gathers its rows in LDS so that they leave as whole cache lines; the
// logarithms of the log-uniform bounds are taken once per block, and the
// normal columns use the noise's logarithm and cosine (gauss.hip).
#define SODECL_SAMPLE_KEY1 0x5EEDD15C0FFEE5EDull
#define SODECL_SAMPLE_CHUNK 120   // its tile of 64 rows stays below 64 KiB
#define SODECL_SAMPLE_WAVES 4

template <int N> struct sodecl_dist_chunk {
    sodecl_dist d[N];
    int c0, nc;   // first column, columns in this chunk
    int groups;   // 64-row groups of a block's tile
    int per;      // columns of a block (blockIdx.y takes the next ones)
};

template <int N> __global__ void __launch_bounds__(64 * SODECL_SAMPLE_WAVES)
sodecl_sample(const sodecl_dist_chunk<N> chunk, int rows, int cols, unsigned long long seed, double* __restrict__ out)
{
    extern __shared__ double sample_lds[];
    const int k0 = (int)blockIdx.y * chunk.per, c0 = chunk.c0 + k0;   // the block's first column
    const int nc = min(chunk.per, chunk.nc - k0), pitch = nc | 1;     // odd: the lanes' rows fall on different banks
    double* const bound = sample_lds;          // per column log a, log b - log a
    double* const tile = sample_lds + 2 * nc;  // [64 * groups][pitch]
    for (int k = threadIdx.x; k < nc; k += blockDim.x) {
        const bool lu = chunk.d[k0 + k].kind == SODECL_DIST_LOG_UNIFORM;
        const double la = lu ? log(chunk.d[k0 + k].a) : 0.0;
        bound[2 * k] = la;
        bound[2 * k + 1] = lu ? log(chunk.d[k0 + k].b) - la : 0.0;
    }
    __syncthreads();
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int tile_rows = 64 * chunk.groups;
    // this thread's entries of a tile in row order: its first, and the distance to the next
    const int first_r = (int)threadIdx.x / nc, first_k = (int)threadIdx.x % nc;
    const int step_r = (int)blockDim.x / nc, step_k = (int)blockDim.x % nc;
    for (long long r0 = (long long)blockIdx.x * tile_rows; r0 < rows; r0 += (long long)gridDim.x * tile_rows) {
        for (int u = wave; u < nc * chunk.groups; u += SODECL_SAMPLE_WAVES) {
            const int k = u / chunk.groups, r = u % chunk.groups * 64 + lane;
            const int kind = chunk.d[k0 + k].kind;
            const double a = chunk.d[k0 + k].a, b = chunk.d[k0 + k].b;
            double v = a;
            if (kind != SODECL_DIST_CONSTANT) {
                sodecl_u64 w0, w1;
                sodecl_threefry2x64_20((sodecl_u64)(r0 + r), (sodecl_u64)(c0 + k), (sodecl_u64)seed,
                                       SODECL_SAMPLE_KEY1, &w0, &w1);
                const double u0 = sodecl_u01(w0);
                if (kind == SODECL_DIST_UNIFORM) {
                    v = fma(b - a, u0, a);
                } else if (kind == SODECL_DIST_LOG_UNIFORM) {
                    v = exp(fma(bound[2 * k + 1], u0, bound[2 * k]));
                } else {   // normal: Box-Muller, cosine branch
                    double s, c;
                    sodecl_sincos_reduced(2.0 * M_PI * sodecl_u01(w1), &s, &c);
                    v = fma(b, sodecl_sqrt_near(-2.0 * sodecl_log_positive(u0)) * c, a);
                }
            }
            tile[r * pitch + k] = v;
        }
        __syncthreads();
        const int here = (int)min((long long)tile_rows, rows - r0);
        for (int r = first_r, k = first_k; r < here;) {
            out[(size_t)(r0 + r) * cols + c0 + k] = tile[r * pitch + k];
            r += step_r;
            k += step_k;
            if (k >= nc) {
                k -= nc;
                ++r;
            }
        }
        __syncthreads();   // before the next tile
    }
}

// Launches columns [c0, c0 + nc) of the table, nc <= N.
template <int N>
static bool sample_chunk(const sodecl_dist* dists, int c0, int nc, int rows, int cols, unsigned long long seed,
                         double* out, int cus, hipStream_t stream)
{
    sodecl_dist_chunk<N> chunk;
    std::memset(&chunk, 0, sizeof chunk);
    chunk.c0 = c0;
    chunk.nc = nc;
    std::memcpy(chunk.d, dists + c0, (size_t)nc * sizeof(sodecl_dist));
    // a narrow chunk takes several 64-row groups per tile, so that each of
    // a block's wavefronts has a few columns' worth of draws between barriers;
    // a table of fewer row groups than SIMDs spreads its columns over blocks
    // instead (down to one column per wavefront), since its time is one
    // wavefront's chain of draws (one call and its completion, 65 columns:
    // 300 rows 32.7 -> 30.4, 17000 rows 46.6 -> 40.4, 30000 rows 47.8 -> 45.1 us)
    const long long row_groups = (rows + 63LL) / 64;
    const bool small = row_groups < 4 * cus;
    chunk.groups = small || nc >= 16 ? 1 : (16 + nc - 1) / nc;
    chunk.per = nc;
    if (small) {
        const long long parts = (4LL * cus + row_groups - 1) / row_groups;
        chunk.per = std::max(std::min(nc, SODECL_SAMPLE_WAVES), (int)((nc + parts - 1) / parts));
    }
    const long long tile_rows = 64LL * chunk.groups;
    const long long blocks = std::min((rows + tile_rows - 1) / tile_rows, (long long)cus * 8);
    const unsigned parts = (unsigned)((nc + chunk.per - 1) / chunk.per);
    const size_t lds = (2 * (size_t)chunk.per + (size_t)tile_rows * (chunk.per | 1)) * sizeof(double);
    hipLaunchKernelGGL(sodecl_sample<N>, dim3((unsigned)blocks, parts), dim3(64 * SODECL_SAMPLE_WAVES), lds, stream,
                       chunk, rows, cols, seed, out);
    return hipGetLastError() == hipSuccess;
}

extern "C" int sodecl_sample_device(const sodecl_dist* dists, int rows, int cols, unsigned long long seed,
                                    double* out, void* stream)
{
    if (!dists || !out || rows < 0 || cols <= 0) return 0;
    for (int c = 0; c < cols; ++c) {
        const sodecl_dist& d = dists[c];
        if (d.kind < SODECL_DIST_CONSTANT || d.kind > SODECL_DIST_NORMAL) return 0;
        if (d.kind == SODECL_DIST_LOG_UNIFORM && !(d.a > 0 && d.b > 0)) return 0;
    }
    if (rows == 0) return 1;
    int device = 0;
    (void)hipGetDevice(&device);
    int cus = 256;
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
    // (the distributions travel in the kernel's arguments, which the host copies
    // at each launch: three sizes, 0.3 us less for 16 columns than for 120)
    for (int c0 = 0; c0 < cols; c0 += SODECL_SAMPLE_CHUNK) {
        const int nc = std::min(cols - c0, SODECL_SAMPLE_CHUNK);
        const hipStream_t s = (hipStream_t)stream;
        const bool ok = nc <= 16   ? sample_chunk<16>(dists, c0, nc, rows, cols, seed, out, cus, s)
                        : nc <= 64 ? sample_chunk<64>(dists, c0, nc, rows, cols, seed, out, cus, s)
                                   : sample_chunk<SODECL_SAMPLE_CHUNK>(dists, c0, nc, rows, cols, seed, out, cus, s);
        if (!ok) return 0;
    }
    return 1;
}
