// A step's small host arrays into their device buffers in one launch.
//
//   vda_upload            up to UPLOAD_MAX blocks of rows, read from mapped pinned memory by the kernel itself
//   vda_mapped_host       where the device sees a pinned allocation
//
// Bound by one trip over the host link and a launch.  us, six arrays of 48 bytes: a copy each 27.3 (27.2 of the host), this 6.3; one array
// of 64 KB 5.2, of 256 KB 8.0 (a copy 13.8), of a megabyte 21.8 (27.7).  A decode step of twelve sequences through four layers of 2048, whose
// block table's columns took a copy and a kernel: 730 -> 650 together with the row index that went up for rows in order.  16 bytes a
// lane where both sides are aligned.
#include "common.h"

constexpr int UPLOAD_MAX = 16;
struct UploadBlock {
  const uint32_t* src;   // dense, in mapped host memory
  uint32_t* dst;
  long width, rows;      // words of a row, rows
  long pitch;            // words between rows of dst
};
struct UploadArgs { UploadBlock block[UPLOAD_MAX]; };

__global__ __launch_bounds__(256) void upload_kernel(const UploadArgs a) {
  const UploadBlock b = a.block[blockIdx.y];
  const long i0 = (long)blockIdx.x * 256 + threadIdx.x, step = (long)gridDim.x * 256;
  if (b.rows == 1 || b.pitch == b.width) {
    const long n = b.width * b.rows;
    const long quads = ((reinterpret_cast<uintptr_t>(b.src) | reinterpret_cast<uintptr_t>(b.dst)) & 15) ? 0 : n >> 2;
    for (long i = i0; i < quads; i += step) reinterpret_cast<u32x4*>(b.dst)[i] = reinterpret_cast<const u32x4*>(b.src)[i];
    for (long i = 4 * quads + i0; i < n; i += step) b.dst[i] = b.src[i];
    return;
  }
  for (long i = i0; i < b.width * b.rows; i += step) {
    const long r = i / b.width;
    b.dst[r * b.pitch + i - r * b.width] = b.src[i];
  }
}

// table: n rows of (source as the device sees it, destination, words of a row, rows, words between rows of the destination), on the host
VDA_EXPORT int vda_upload(const long* table, int n, hipStream_t st) {
  if (n < 1 || n > UPLOAD_MAX) return n == 0 ? 0 : -1;
  UploadArgs a = {};
  long most = 0;
  for (int i = 0; i < n; ++i) {
    const long* t = table + 5 * i;
    if (!t[0] || !t[1] || t[0] % 4 || t[1] % 4 || t[2] < 1 || t[3] < 1 || (t[3] > 1 && t[4] < t[2])) return -1;
    a.block[i] = UploadBlock{reinterpret_cast<const uint32_t*>(t[0]), reinterpret_cast<uint32_t*>(t[1]), t[2], t[3], t[4]};
    if (t[2] * t[3] > most) most = t[2] * t[3];
  }
  const long groups = (most + 1023) / 1024;
  hipLaunchKernelGGL(upload_kernel, dim3((unsigned)(groups < 64 ? groups : 64), n), dim3(256), 0, st, a);
  VDA_CHECK_LAUNCH();
  return 0;
}

VDA_EXPORT int vda_mapped_host(void** device, void* host) {
  return (int)hipHostGetDevicePointer(device, host, 0);
}
