// tq_cache_grow.hip -- one launch that fills a cache layer's new buffers on
// growth (CompressedStorage::ensure_capacity, reference
// src/cache/storage.rs:108-139, and ensure_qjl_capacity, src/cache/tq.rs:64-94):
// the stored rows copied from the old buffers, the rest zero as Tensor::zeros.
//
// Every byte of the new buffers is written once, and the old rows are read
// once.  What it replaces was bound by launches and host calls, not bytes: a
// fill per buffer and a strided copy per buffer, 8 to 12 operations of about
// 2 us on the GPU and 2.4 to 3.2 us on the host each.
#include "tq_common.h"

#include <algorithm>

namespace {

struct GrowArgs {
  tqh::GrowPart part[tqh::kGrowParts];
  long long old_cap, new_cap, rows;  // records per head: old pitch, new pitch, stored
  int heads;
};

template <class T>
__device__ void grow(const tqh::GrowPart &p, const GrowArgs &a) {
  const long long per = p.rec_bytes / (int)sizeof(T);
  const long long used = a.rows * per, pitch = a.new_cap * per, old_pitch = a.old_cap * per;
  const T *src = static_cast<const T *>(p.src);
  T *dst = static_cast<T *>(p.dst);
  for (long long h = blockIdx.y; h < a.heads; h += gridDim.y)
    for (long long u = (long long)blockIdx.x * blockDim.x + threadIdx.x; u < pitch; u += (long long)gridDim.x * blockDim.x)
      dst[h * pitch + u] = u < used ? src[h * old_pitch + u] : T{};
}

// One buffer per z.  Records are of even size and every buffer starts on a
// 16-byte boundary, so the widest unit that divides a record divides every
// offset.
__global__ __launch_bounds__(256) void cache_grow_kernel(GrowArgs a) {
  const tqh::GrowPart p = a.part[blockIdx.z];
  if (p.rec_bytes % 16 == 0) grow<uint4>(p, a);
  else if (p.rec_bytes % 8 == 0) grow<uint2>(p, a);
  else if (p.rec_bytes % 4 == 0) grow<uint32_t>(p, a);
  else grow<uint16_t>(p, a);
}

}  // namespace

namespace tqh {

int grow_layer(const GrowPart *parts, int num_parts, int heads, long long old_cap, long long new_cap, long long rows,
               hipStream_t stream) {
  GrowArgs a{};
  long long units = 1;
  for (int i = 0; i < num_parts; i++) {
    a.part[i] = parts[i];
    int u = 16;
    while (parts[i].rec_bytes % u) u /= 2;
    units = std::max(units, new_cap * (parts[i].rec_bytes / u));
  }
  a.old_cap = old_cap;
  a.new_cap = new_cap;
  a.rows = rows;
  a.heads = heads;
  const dim3 grid((unsigned)std::min<long long>((units + 255) / 256, 1024), (unsigned)std::min(heads, 65535),
                  (unsigned)num_parts);
  hipLaunchKernelGGL(cache_grow_kernel, grid, dim3(256), 0, stream, a);
  return check_launch("cache_grow_kernel");
}

}  // namespace tqh
