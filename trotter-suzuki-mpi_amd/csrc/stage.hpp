// stage.hpp -- host arrays of a state to and from its device planes.
//
// The copies of the runtime from and to ordinary host memory register the pages
// of every call's array with the GPU and release them after it (2 x 1032^2
// complex in FP32, up and down: 77 ms of a call whose 1000 steps take 30 ms).
// Here the rows pass through two pinned chunks that the owner keeps: the CPU
// copies one while a kernel reads or writes the other over the host link,
// taking the pair of planes apart (or interleaving it), rounding once on the way
// in and dividing by a pending renormalisation on the way out, so no host pass
// does either and no temporary array is made.
//
// Host arrays are two planes of doubles (re, im) or one of complex doubles
// (im == nullptr: re points at interleaved values).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

namespace tsmi {

template <typename T>
__global__ void stage_in_kernel(const double *__restrict__ src, T *__restrict__ re, T *__restrict__ im, int w,
                                int rows, long pitch, int interleaved) {
    const int n = w * rows;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int y = i / w;
        const long d = y * pitch + (i - y * w);
        if (interleaved) {
            const double2 z = reinterpret_cast<const double2 *>(src)[i];
            re[d] = (T)z.x;
            im[d] = (T)z.y;
        } else {
            re[d] = (T)src[i];
            im[d] = (T)src[n + i];
        }
    }
}

template <typename T>
__global__ void stage_out_kernel(const T *__restrict__ re, const T *__restrict__ im, double *__restrict__ dst, int w,
                                 int rows, long pitch, int interleaved, const double *__restrict__ div) {
    const int n = w * rows;
    const double d = div ? *div : 1.0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int y = i / w;
        const long s = y * pitch + (i - y * w);
        double vr = (double)re[s], vi = (double)im[s];
        if (div) {
            vr /= d;
            vi /= d;
        }
        if (interleaved) {
            reinterpret_cast<double2 *>(dst)[i] = make_double2(vr, vi);
        } else {
            dst[i] = vr;
            dst[n + i] = vi;
        }
    }
}

// Two pinned chunks of at most kChunk bytes each (or one row, if that is more), allocated at the first use and
// released with the owner.  A call returns when its copies are done, so the
// chunks are free between calls, whatever stream the next one runs on.
class HostStage {
  public:
    HostStage() = default;
    HostStage(const HostStage &) = delete;
    HostStage &operator=(const HostStage &) = delete;
    ~HostStage() { release(); }

    void release() {
        for (int k = 0; k < 2; ++k) {
            if (buf_[k]) (void)hipHostFree(buf_[k]);
            if (ev_[k]) (void)hipEventDestroy(ev_[k]);
            buf_[k] = nullptr;
            ev_[k] = nullptr;
        }
        cap_ = 0;
    }

    // w x h values of row stride `stride` into planes of row pitch `pitch`
    template <typename T>
    hipError_t upload(hipStream_t s, T *re, T *im, long pitch, const double *hre, const double *him, size_t w,
                      size_t h, size_t stride) {
        size_t rows = 0;
        hipError_t e = reserve(w, h, &rows);
        for (size_t y = 0, k = 0; y < h && e == hipSuccess; y += rows, k ^= 1) {
            const size_t m = std::min(rows, h - y);
            if (y >= 2 * rows) e = hipEventSynchronize(ev_[k]);   // the chunk's last reader
            if (e != hipSuccess) break;
            const int z = him ? 0 : 1;
            copy_rows(buf_[k], w << z, hre + ((y * stride) << z), stride << z, w << z, m);
            if (him) copy_rows(buf_[k] + w * m, w, him + y * stride, stride, w, m);
            hipLaunchKernelGGL((stage_in_kernel<T>), dim3(blocks(w * m)), dim3(256), 0, s, (const double *)buf_[k],
                               re + (long)y * pitch, im + (long)y * pitch, (int)w, (int)m, pitch, z);
            e = hipGetLastError();
            if (e == hipSuccess) e = hipEventRecord(ev_[k], s);
        }
        const hipError_t f = hipStreamSynchronize(s);
        return e != hipSuccess ? e : f;
    }

    // the reverse; *div (device memory, may be null) divides every value
    template <typename T>
    hipError_t download(hipStream_t s, const T *re, const T *im, long pitch, double *hre, double *him, size_t w,
                        size_t h, size_t stride, const double *div) {
        size_t rows = 0;
        hipError_t e = reserve(w, h, &rows);
        const int z = him ? 0 : 1;
        auto launch = [&](size_t y, size_t k) {
            const size_t m = std::min(rows, h - y);
            hipLaunchKernelGGL((stage_out_kernel<T>), dim3(blocks(w * m)), dim3(256), 0, s, re + (long)y * pitch,
                               im + (long)y * pitch, buf_[k], (int)w, (int)m, pitch, z, div);
            const hipError_t f = hipGetLastError();
            return f != hipSuccess ? f : hipEventRecord(ev_[k], s);
        };
        if (e == hipSuccess && h > 0) e = launch(0, 0);
        for (size_t y = 0, k = 0; y < h && e == hipSuccess; y += rows, k ^= 1) {
            const size_t m = std::min(rows, h - y);
            if (y + rows < h) e = launch(y + rows, k ^ 1);
            if (e == hipSuccess) e = hipEventSynchronize(ev_[k]);
            if (e != hipSuccess) break;
            copy_rows(hre + ((y * stride) << z), stride << z, buf_[k], w << z, w << z, m);
            if (him) copy_rows(him + y * stride, stride, buf_[k] + w * m, w, w, m);
        }
        const hipError_t f = hipStreamSynchronize(s);
        return e != hipSuccess ? e : f;
    }

  private:
    static constexpr size_t kChunk = 4u << 20;

    static int blocks(size_t n) { return (int)std::min<size_t>(512, (n + 255) / 256); }

    static void copy_rows(double *d, size_t dstride, const double *s, size_t sstride, size_t w, size_t rows) {
        if (dstride == w && sstride == w) {
            std::memcpy(d, s, rows * w * sizeof(double));
            return;
        }
        for (size_t y = 0; y < rows; ++y) std::memcpy(d + y * dstride, s + y * sstride, w * sizeof(double));
    }

    // chunks for w-wide rows: *rows of them per chunk
    hipError_t reserve(size_t w, size_t h, size_t *rows) {
        const size_t row = 2 * w * sizeof(double);
        *rows = std::max<size_t>(1, std::min(h, kChunk / row));
        // a state of one chunk's size is cut in two, so that the halves overlap
        if (*rows == h && h > 1 && h * row > (256u << 10)) *rows = (h + 1) / 2;
        const size_t need = *rows * row;
        hipError_t e = hipSuccess;
        if (need > cap_) {
            release();
            for (int k = 0; k < 2 && e == hipSuccess; ++k) {
                e = hipHostMalloc((void **)&buf_[k], need, hipHostMallocDefault);
                if (e == hipSuccess) e = hipEventCreateWithFlags(&ev_[k], hipEventDisableTiming);
            }
            if (e != hipSuccess) {
                release();
                return e;
            }
            cap_ = need;
        }
        return e;
    }

    double *buf_[2] = {nullptr, nullptr};
    hipEvent_t ev_[2] = {nullptr, nullptr};
    size_t cap_ = 0;
};

}  // namespace tsmi
