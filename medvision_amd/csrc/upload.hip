// Small host arrays to device memory without a copy engine: the bytes travel as kernel arguments.
//
// The augmentation stages send a few rois (40 bytes each) or a control grid (6 KB) per call.  A copy from
// pageable memory waits for everything queued on the stream, so that every stage of a pipeline ended in an idle GPU
// (five of them in one resize / affine / elastic / crop chain: 15 - 20 us each, 0.37 ms for the chain); a copy from
// pinned memory costs ~10 us of host time and a blit launch.  A launch with the bytes in its argument block is
// asynchronous, needs no staging buffer whose lifetime someone has to watch, and takes ~3 us.
#include "common.hpp"

#include <cstring>

namespace mv {

// (kernel arguments are limited to 4 KB)
constexpr int kUploadWords = 960;
struct UploadBlock {
  unsigned words[kUploadWords];
};

__global__ void __launch_bounds__(256) upload_kernel(UploadBlock block, unsigned *__restrict__ out, int words) {
  for (int i = threadIdx.x; i < words; i += 256) out[i] = block.words[i];
}

}  // namespace mv

extern "C" int mv_upload(const void *host, void *device, size_t bytes, void *stream) {
  MV_REQUIRE(bytes % 4 == 0 && reinterpret_cast<uintptr_t>(device) % 4 == 0, "whole 4-byte words are uploaded");
  if (bytes == 0) return MV_OK;
  MV_REQUIRE(host && device, "null pointer argument");
  MV_REQUIRE(bytes <= MV_UPLOAD_MAX_BYTES, "mv_upload is for at most %zu bytes", static_cast<size_t>(MV_UPLOAD_MAX_BYTES));
  const char *src = static_cast<const char *>(host);
  unsigned *dst = static_cast<unsigned *>(device);
  for (size_t left = bytes; left > 0;) {
    mv::UploadBlock block;
    const size_t part = left < sizeof(block) ? left : sizeof(block);
    std::memcpy(block.words, src, part);
    hipLaunchKernelGGL(mv::upload_kernel, dim3(1), dim3(256), 0, static_cast<hipStream_t>(stream), block, dst,
                       static_cast<int>(part / 4));
    src += part;
    dst += part / 4;
    left -= part;
  }
  return mv::check_launch("upload_kernel");
}
