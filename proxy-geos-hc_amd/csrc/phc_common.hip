// phc_common.hip -- error text, device buffers and library-wide entry points.
#include "phc_common.hpp"
#include "readback.hpp"

#include <algorithm>
#include <vector>

namespace phc {

static thread_local std::string g_last_error = "no error";

void set_error(const char *fmt, ...)
{
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_last_error = buf;
}

phc_status fail(phc_status code, const char *fmt, ...)
{
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_last_error = buf;
    return code;
}

phc_status DevBuf::alloc(size_t n)
{
    release();
    if (n == 0) return PHC_OK;
    hipError_t e = hipMalloc(&ptr, n);
    if (e != hipSuccess) {
        ptr = nullptr;
        return fail(e == hipErrorOutOfMemory ? PHC_ERR_NOMEM : PHC_ERR_HIP,
                    "hipMalloc(%zu) failed: %s", n, hipGetErrorString(e));
    }
    bytes = n;
    return PHC_OK;
}

void DevBuf::release()
{
    if (ptr) (void)hipFree(ptr);
    ptr = nullptr;
    bytes = 0;
}

} // namespace phc

extern "C" {

const char *phc_last_error(void) { return phc::g_last_error.c_str(); }

const char *phc_version(void) { return "phc 0.1 gfx950"; }

int phc_device_count(void)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

phc_status phc_device_synchronize(void)
{
    PHC_HIP(hipDeviceSynchronize());
    return PHC_OK;
}

} // extern "C"

// ---------------------------------------------------------------------------
// Reading fields back (readback.hpp)
namespace phc {

// Face-slab rule of the sponge at interior point (i, j, k).
__host__ __device__ inline float face_damping(int sw, const float *fx, const float *fy, const float *fz,
                                              const FdLayout &L, int i, int j, int k)
{
    const bool inI = i >= sw && i < L.nx - sw, inJ = j >= sw && j < L.ny - sw, inK = k >= sw && k < L.nz - sw;
    float s = 1.f;
    if (inJ && inK && !inI) s = fx[i];
    if (inK && inI && !inJ) s = fy[j];
    if (inJ && inI && !inK) s = fz[k];
    return s;
}

// `rows` rows of the field from row r0 on (rows along k, planes after each
// other); four rows per block, 64 lanes along a row.
static __global__ void __launch_bounds__(256)
pack_rows_kernel(const float *p, FdLayout L, int r0, int rows, int lx, int ly, int lz, FieldDamping d, float *out)
{
    const int row = blockIdx.x * 4 + threadIdx.y, NY = L.ny + 2 * ly, NZ = L.nz + 2 * lz;
    if (row >= rows) return;
    const int i = (r0 + row) / NY - lx, j = (r0 + row) % NY - ly;
    const float *src = p + fd_off(L, i, j, -lz);
    float *dst = out + (int64_t)row * NZ;
    const bool damp = d.sw > 0 && i >= 0 && i < L.nx && j >= 0 && j < L.ny;
    for (int c = threadIdx.x; c < NZ; c += 64) {
        float v = src[c];
        const int k = c - lz;
        if (damp && k >= 0 && k < L.nz) v *= face_damping(d.sw, d.fx, d.fy, d.fz, L, i, j, k);
        dst[c] = v;
    }
}

static __global__ void __launch_bounds__(256)
unpack_rows_kernel(float *p, FdLayout L, int r0, int rows, int lx, int ly, int lz, const float *in)
{
    const int row = blockIdx.x * 4 + threadIdx.y, NY = L.ny + 2 * ly, NZ = L.nz + 2 * lz;
    if (row >= rows) return;
    float *dst = p + fd_off(L, (r0 + row) / NY - lx, (r0 + row) % NY - ly, -lz);
    const float *src = in + (int64_t)row * NZ;
    for (int c = threadIdx.x; c < NZ; c += 64) dst[c] = src[c];
}

static __global__ void __launch_bounds__(256) fill_field_kernel(float *p, int64_t n, float v)
{
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < n; t += stride) p[t] = v;
}

// Rows k0 .. k0 + n - 1 of the slice; 64 points along k by 4 along i per block:
// reads run along k.
static __global__ void __launch_bounds__(256)
slice_xz_kernel(const float *p, FdLayout L, int j, int k0, int n, FieldDamping d, float *out)
{
    const int r = blockIdx.x * 64 + threadIdx.x, i = blockIdx.y * 4 + threadIdx.y, k = k0 + r;
    if (r >= n || i >= L.nx) return;
    float v = p[fd_off(L, i, j, k)];
    if (d.sw > 0) v *= face_damping(d.sw, d.fx, d.fy, d.fz, L, i, j, k);
    out[(int64_t)r * L.nx + i] = v;
}

static bool ensure_scratch(DevBuf &b, size_t bytes)
{
    if (b.bytes >= bytes) return true;
    if (b.alloc(bytes) == PHC_OK) return true;
    (void)hipGetLastError();
    return false;
}

// Rows of NZ floats that a piece of at most READ_PIECE bytes holds.
static int piece_rows(int rows, int NZ)
{
    return (int)std::min<size_t>(rows, std::max<size_t>(1, READ_PIECE / (sizeof(float) * (size_t)NZ)));
}

phc_status read_field(hipStream_t stream, DevBuf &scratch, const float *field, const FdLayout &L, int lx, int ly,
                      int lz, const FieldDamping &damping, const float *const host_factors[3], float *host)
{
    const int NX = L.nx + 2 * lx, NY = L.ny + 2 * ly, NZ = L.nz + 2 * lz, rows = NX * NY;
    const size_t row = sizeof(float) * (size_t)NZ;
    const int per = piece_rows(rows, NZ);
    if (!ensure_scratch(scratch, row * per)) {
        PHC_HIP(hipStreamSynchronize(stream));
        for (int i = 0; i < NX; ++i) {
            float *plane = host + (int64_t)i * NY * NZ;
            PHC_HIP(hipMemcpy2D(plane, row, field + fd_off(L, i - lx, -ly, -lz), sizeof(float) * L.pitch_k, row, NY,
                                hipMemcpyDeviceToHost));
            if (damping.sw <= 0 || i < lx || i >= lx + L.nx) continue;
            for (int j = 0; j < L.ny; ++j)
                for (int k = 0; k < L.nz; ++k)
                    plane[(int64_t)(j + ly) * NZ + k + lz] *= face_damping(
                        damping.sw, host_factors[0], host_factors[1], host_factors[2], L, i - lx, j, k);
        }
        return PHC_OK;
    }
    for (int r0 = 0; r0 < rows; r0 += per) {
        const int n = std::min(per, rows - r0);
        hipLaunchKernelGGL(pack_rows_kernel, dim3((n + 3) / 4), dim3(64, 4), 0, stream, field, L, r0, n, lx, ly, lz,
                           damping, scratch.as<float>());
        PHC_HIP(hipGetLastError());
        PHC_HIP(hipMemcpyAsync(host + (int64_t)r0 * NZ, scratch.ptr, row * n, hipMemcpyDeviceToHost, stream));
    }
    PHC_HIP(hipStreamSynchronize(stream));
    return PHC_OK;
}

phc_status write_field(hipStream_t stream, DevBuf &scratch, float *field, const FdLayout &L, int lx, int ly, int lz,
                       const float *host)
{
    const int NX = L.nx + 2 * lx, NY = L.ny + 2 * ly, NZ = L.nz + 2 * lz, rows = NX * NY;
    const size_t row = sizeof(float) * (size_t)NZ;
    const int per = piece_rows(rows, NZ);
    PHC_HIP(hipStreamSynchronize(stream));
    if (!ensure_scratch(scratch, row * per)) {
        for (int i = 0; i < NX; ++i)
            PHC_HIP(hipMemcpy2D(field + fd_off(L, i - lx, -ly, -lz), sizeof(float) * L.pitch_k,
                                host + (int64_t)i * NY * NZ, row, row, NY, hipMemcpyHostToDevice));
        return PHC_OK;
    }
    for (int r0 = 0; r0 < rows; r0 += per) {
        const int n = std::min(per, rows - r0);
        // a plain copy: the first large asynchronous copy on a stream sets up
        // staging memory, which would add 4 ms to every create
        PHC_HIP(hipMemcpy(scratch.ptr, host + (int64_t)r0 * NZ, row * n, hipMemcpyHostToDevice));
        hipLaunchKernelGGL(unpack_rows_kernel, dim3((n + 3) / 4), dim3(64, 4), 0, stream, field, L, r0, n, lx, ly, lz,
                           scratch.as<float>());
        PHC_HIP(hipGetLastError());
        PHC_HIP(hipStreamSynchronize(stream));  // the next piece overwrites the scratch
    }
    return PHC_OK;
}

phc_status fill_field(hipStream_t stream, float *field, int64_t n, float value)
{
    hipLaunchKernelGGL(fill_field_kernel, dim3((unsigned)std::min<int64_t>((n + 255) / 256, 8192)), dim3(256), 0,
                       stream, field, n, value);
    PHC_HIP(hipGetLastError());
    return PHC_OK;
}

phc_status read_slice_xz(hipStream_t stream, DevBuf &scratch, const float *field, const FdLayout &L, int j,
                         const FieldDamping &damping, const float *const host_factors[3], float *host)
{
    const size_t row = sizeof(float) * (size_t)L.nx;
    const int per = piece_rows(L.nz, L.nx);
    if (!ensure_scratch(scratch, row * per)) {
        PHC_HIP(hipStreamSynchronize(stream));
        std::vector<float> buf((size_t)L.nx * L.nz);
        PHC_HIP(hipMemcpy2D(buf.data(), sizeof(float) * L.nz, field + fd_off(L, 0, j, 0), sizeof(float) * L.pitch_j,
                            sizeof(float) * L.nz, L.nx, hipMemcpyDeviceToHost));
        for (int i = 0; i < L.nx; ++i)
            for (int k = 0; k < L.nz; ++k) {
                float v = buf[(size_t)i * L.nz + k];
                if (damping.sw > 0)
                    v *= face_damping(damping.sw, host_factors[0], host_factors[1], host_factors[2], L, i, j, k);
                host[(int64_t)k * L.nx + i] = v;
            }
        return PHC_OK;
    }
    for (int k0 = 0; k0 < L.nz; k0 += per) {
        const int n = std::min(per, L.nz - k0);
        hipLaunchKernelGGL(slice_xz_kernel, dim3((n + 63) / 64, (L.nx + 3) / 4), dim3(64, 4), 0, stream, field, L, j,
                           k0, n, damping, scratch.as<float>());
        PHC_HIP(hipGetLastError());
        PHC_HIP(hipMemcpyAsync(host + (int64_t)k0 * L.nx, scratch.ptr, row * n, hipMemcpyDeviceToHost, stream));
    }
    PHC_HIP(hipStreamSynchronize(stream));
    return PHC_OK;
}

} // namespace phc

// ---------------------------------------------------------------------------
// Bandwidth calibration: a plain streaming copy of known size, used to scale
// the HBM byte counters (FETCH_SIZE / WRITE_SIZE) of the stencil kernels and
// to state the practical copy bandwidth beside the 8 TB/s peak.
__global__ void phc_copy_kernel(const float4 *__restrict__ src, float4 *__restrict__ dst, size_t n)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) dst[i] = src[i];
}

extern "C" phc_status phc_copy_bandwidth(size_t bytes, int iters, double *ms_per_copy)
{
    if (!ms_per_copy || iters < 1 || bytes < 16)
        return phc::fail(PHC_ERR_INVALID, "bad copy-bandwidth arguments");
    const size_t n = bytes / 16;
    phc::DevBuf a, b;
    PHC_TRY(a.alloc(n * 16));
    PHC_TRY(b.alloc(n * 16));
    PHC_HIP(hipMemset(a.ptr, 0, n * 16));
    hipEvent_t e0, e1;
    PHC_HIP(hipEventCreate(&e0));
    PHC_HIP(hipEventCreate(&e1));
    const int blocks = 256 * 8;
    hipLaunchKernelGGL(phc_copy_kernel, dim3(blocks), dim3(256), 0, 0, a.as<float4>(), b.as<float4>(), n);
    PHC_HIP(hipEventRecord(e0, 0));
    for (int it = 0; it < iters; ++it)
        hipLaunchKernelGGL(phc_copy_kernel, dim3(blocks), dim3(256), 0, 0, a.as<float4>(),
                           b.as<float4>(), n);
    PHC_HIP(hipEventRecord(e1, 0));
    PHC_HIP(hipEventSynchronize(e1));
    float ms = 0.f;
    PHC_HIP(hipEventElapsedTime(&ms, e0, e1));
    *ms_per_copy = ms / iters;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return PHC_OK;
}
