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

// Four rows per block, 64 lanes along a row.
static __global__ void __launch_bounds__(256)
pack_rows_kernel(const float *p, FdLayout L, int i0, int rows, int ly, int lz, FieldDamping d, float *out)
{
    const int row = blockIdx.x * 4 + threadIdx.y, NY = L.ny + 2 * ly, NZ = L.nz + 2 * lz;
    if (row >= rows) return;
    const int i = i0 + row / NY, j = row % NY - ly;
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
unpack_rows_kernel(float *p, FdLayout L, int i0, int rows, int ly, int lz, const float *in)
{
    const int row = blockIdx.x * 4 + threadIdx.y, NY = L.ny + 2 * ly, NZ = L.nz + 2 * lz;
    if (row >= rows) return;
    float *dst = p + fd_off(L, i0 + row / NY, row % NY - ly, -lz);
    const float *src = in + (int64_t)row * NZ;
    for (int c = threadIdx.x; c < NZ; c += 64) dst[c] = src[c];
}

static __global__ void __launch_bounds__(256) fill_field_kernel(float *p, int64_t n, float v)
{
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < n; t += stride) p[t] = v;
}

// 64 points along k by 4 along i per block: reads run along k.
static __global__ void __launch_bounds__(256)
slice_xz_kernel(const float *p, FdLayout L, int j, FieldDamping d, float *out)
{
    const int k = blockIdx.x * 64 + threadIdx.x, i = blockIdx.y * 4 + threadIdx.y;
    if (k >= L.nz || i >= L.nx) return;
    float v = p[fd_off(L, i, j, k)];
    if (d.sw > 0) v *= face_damping(d.sw, d.fx, d.fy, d.fz, L, i, j, k);
    out[(int64_t)k * L.nx + i] = v;
}

static bool ensure_scratch(DevBuf &b, size_t bytes)
{
    if (b.bytes >= bytes) return true;
    if (b.alloc(bytes) == PHC_OK) return true;
    (void)hipGetLastError();
    return false;
}

phc_status read_field(hipStream_t stream, DevBuf &scratch, const float *field, const FdLayout &L, int lx, int ly,
                      int lz, const FieldDamping &damping, const float *const host_factors[3], float *host)
{
    const int NX = L.nx + 2 * lx, NY = L.ny + 2 * ly, NZ = L.nz + 2 * lz;
    const size_t plane = sizeof(float) * (size_t)NY * NZ;
    // floats from a plane's first value to its last
    const int64_t span = (int64_t)(NY - 1) * L.pitch_k + NZ;
    const int per = (int)std::min<size_t>(NX, std::max<size_t>(1, READ_PIECE / plane));
    if (!ensure_scratch(scratch, plane * per)) {
        PHC_HIP(hipStreamSynchronize(stream));
        std::vector<float> buf((size_t)((per - 1) * L.pitch_j + span));
        for (int i0 = 0; i0 < NX; i0 += per) {
            const int n = std::min(per, NX - i0);
            PHC_HIP(hipMemcpy(buf.data(), field + fd_off(L, i0 - lx, -ly, -lz),
                              sizeof(float) * (size_t)((n - 1) * L.pitch_j + span), hipMemcpyDeviceToHost));
            for (int i = i0; i < i0 + n; ++i)
                for (int j = 0; j < NY; ++j) {
                    float *dst = host + ((int64_t)i * NY + j) * NZ;
                    const float *src = buf.data() + (i - i0) * L.pitch_j + j * L.pitch_k;
                    std::copy(src, src + NZ, dst);
                    if (damping.sw > 0 && i >= lx && i < lx + L.nx && j >= ly && j < ly + L.ny)
                        for (int k = 0; k < L.nz; ++k)
                            dst[k + lz] *= face_damping(damping.sw, host_factors[0], host_factors[1],
                                                        host_factors[2], L, i - lx, j - ly, k);
                }
        }
        return PHC_OK;
    }
    for (int i = 0; i < NX; i += per) {
        const int rows = std::min(per, NX - i) * NY;
        hipLaunchKernelGGL(pack_rows_kernel, dim3((rows + 3) / 4), dim3(64, 4), 0, stream, field, L, i - lx, rows, ly,
                           lz, damping, scratch.as<float>());
        PHC_HIP(hipGetLastError());
        PHC_HIP(hipMemcpyAsync(host + (int64_t)i * NY * NZ, scratch.ptr, sizeof(float) * (size_t)rows * NZ,
                               hipMemcpyDeviceToHost, stream));
    }
    PHC_HIP(hipStreamSynchronize(stream));
    return PHC_OK;
}

phc_status write_field(hipStream_t stream, DevBuf &scratch, float *field, const FdLayout &L, int lx, int ly, int lz,
                       const float *host)
{
    const int NX = L.nx + 2 * lx, NY = L.ny + 2 * ly, NZ = L.nz + 2 * lz;
    const size_t plane = sizeof(float) * (size_t)NY * NZ;
    const int64_t span = (int64_t)(NY - 1) * L.pitch_k + NZ;
    const int per = (int)std::min<size_t>(NX, std::max<size_t>(1, READ_PIECE / plane));
    PHC_HIP(hipStreamSynchronize(stream));
    const bool packed = ensure_scratch(scratch, plane * per);
    std::vector<float> buf(packed ? 0 : (size_t)((per - 1) * L.pitch_j + span));
    for (int i0 = 0; i0 < NX; i0 += per) {
        const int n = std::min(per, NX - i0);
        const float *src = host + (int64_t)i0 * NY * NZ;
        if (packed) {
            PHC_HIP(hipMemcpy(scratch.ptr, src, plane * n, hipMemcpyHostToDevice));
            hipLaunchKernelGGL(unpack_rows_kernel, dim3((n * NY + 3) / 4), dim3(64, 4), 0, stream, field, L, i0 - lx,
                               n * NY, ly, lz, scratch.as<float>());
            PHC_HIP(hipGetLastError());
            PHC_HIP(hipStreamSynchronize(stream));  // the next piece overwrites the scratch
            continue;
        }
        float *dev = field + fd_off(L, i0 - lx, -ly, -lz);
        const size_t bytes = sizeof(float) * (size_t)((n - 1) * L.pitch_j + span);
        PHC_HIP(hipMemcpy(buf.data(), dev, bytes, hipMemcpyDeviceToHost));
        for (int i = 0; i < n; ++i)
            for (int j = 0; j < NY; ++j)
                std::copy(src + ((int64_t)i * NY + j) * NZ, src + ((int64_t)i * NY + j + 1) * NZ,
                          buf.data() + i * L.pitch_j + j * L.pitch_k);
        PHC_HIP(hipMemcpy(dev, buf.data(), bytes, hipMemcpyHostToDevice));
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
    const size_t bytes = sizeof(float) * (size_t)L.nx * L.nz;
    if (!ensure_scratch(scratch, bytes)) {
        PHC_HIP(hipStreamSynchronize(stream));
        std::vector<float> row((size_t)L.nz);
        for (int i = 0; i < L.nx; ++i) {
            PHC_HIP(hipMemcpy(row.data(), field + fd_off(L, i, j, 0), sizeof(float) * L.nz, hipMemcpyDeviceToHost));
            for (int k = 0; k < L.nz; ++k) {
                float v = row[k];
                if (damping.sw > 0)
                    v *= face_damping(damping.sw, host_factors[0], host_factors[1], host_factors[2], L, i, j, k);
                host[(int64_t)k * L.nx + i] = v;
            }
        }
        return PHC_OK;
    }
    hipLaunchKernelGGL(slice_xz_kernel, dim3((L.nz + 63) / 64, (L.nx + 3) / 4), dim3(64, 4), 0, stream, field, L, j,
                       damping, scratch.as<float>());
    PHC_HIP(hipGetLastError());
    PHC_HIP(hipMemcpyAsync(host, scratch.ptr, bytes, hipMemcpyDeviceToHost, stream));
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
