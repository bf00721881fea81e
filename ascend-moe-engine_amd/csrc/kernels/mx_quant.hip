// Standalone block-32 MX quantisation of bf16 rows: the operator behind the reference's stages
// `attn_quant` and `shared_act_quant` (aclnnDynamicMxQuant, src/pipeline/pipeline.cpp:251-258).
// HBM-bound: 2 bytes read, 1 + 1/32 written per element.
#include "kernels.h"
#include "mx_quant_device.h"

namespace mlakv {
namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

constexpr int kThreads = 256;

// An item is 8 consecutive values (16 bytes in, 8 bytes out); the four items of a block of 32 belong
// to neighbouring lanes of one wavefront (cols is a multiple of 32, so blocks never straddle rows).
// The items of all rows, end to end, are dealt to workgroups 256 x LOADS at a time; a thread asks for
// its LOADS items before it uses the first.
// What bounds it is HBM, once the arithmetic and the addresses are short: with one item per thread,
// each dividing its 64-bit item number by the row length, a large launch was bound by its vector
// instructions. Measured per launch, rows of 64 x 512 values: 4096 rows 75.9 -> 63.7 us (6.3 TB/s),
// 300 rows 7.8 -> 7.6 us, 32 rows 2.75 -> 2.56 us.
// GROUPED: rows in groups with strides of their own, a division more per item.
template <int LOADS, bool GROUPED>
__global__ __launch_bounds__(kThreads) void MxQuantKernel(MxQuantArgs q) {
  const auto at_row = [&](int64_t row, int64_t row_stride, int64_t group_stride) __attribute__((always_inline)) {
    if constexpr (!GROUPED) return row * row_stride;
    const unsigned group = static_cast<unsigned>(row) / static_cast<unsigned>(q.group_rows);  // (fewer than 2^32 rows, ensured by the launcher)
    return group * group_stride + (row - static_cast<int64_t>(group) * q.group_rows) * row_stride;
  };
  constexpr int kItemsPerGroup = kThreads * LOADS;
  const unsigned items_per_row = static_cast<unsigned>(q.cols) >> 3;
  // the workgroup's first item: a division on uniform values, in 32 bits wherever they suffice
  const int64_t first = static_cast<int64_t>(blockIdx.x) * kItemsPerGroup;
  const int64_t row0 = first <= 0x7fffffff ? static_cast<unsigned>(first) / items_per_row : first / items_per_row;
  const unsigned col0 = static_cast<unsigned>(first - row0 * items_per_row);
  u32x4 v[LOADS];
  int64_t row[LOADS];
  unsigned col[LOADS];  // in items
  bool live[LOADS];     // dead lanes still take part in the exchanges
#pragma unroll
  for (int u = 0; u < LOADS; ++u) {
    const unsigned at = col0 + threadIdx.x + kThreads * u;
    // rows of at least kItemsPerGroup items: the workgroup's items end in the row behind the first at the latest
    const unsigned ahead = items_per_row >= kItemsPerGroup ? (at >= items_per_row ? 1u : 0u) : at / items_per_row;
    row[u] = row0 + ahead;
    col[u] = at - ahead * items_per_row;
    live[u] = row[u] < q.rows;
    v[u] = u32x4{0u, 0u, 0u, 0u};
    if (live[u]) v[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(q.x + at_row(row[u], q.x_row_stride, q.x_group_stride) + col[u] * 16));
  }
#pragma unroll
  for (int u = 0; u < LOADS; ++u) {
    unsigned magnitude = 0u;
#pragma unroll
    for (int i = 0; i < 4; ++i) magnitude = MxMagnitudeMax(v[u][i], magnitude);
    magnitude = max(magnitude, static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, static_cast<int>(magnitude), 0xb1, 0xf, 0xf, false)));  // quad_perm:[1,0,3,2]
    magnitude = max(magnitude, static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, static_cast<int>(magnitude), 0x4e, 0xf, 0xf, false)));  // quad_perm:[2,3,0,1]
    if (!live[u]) continue;
    const MxScale s = MxScaleFromMaxBits(magnitude);
    const u32x2 codes = {MxEncodeFour(v[u][0], v[u][1], s), MxEncodeFour(v[u][2], v[u][3], s)};
    __builtin_nontemporal_store(codes, reinterpret_cast<u32x2*>(q.codes + at_row(row[u], q.codes_row_stride, q.codes_group_stride) + col[u] * 8));
    if ((col[u] & 3u) == 0u) {
      reinterpret_cast<unsigned char*>(q.scales + at_row(row[u], q.scales_row_stride, q.scales_group_stride))[col[u] >> 2] = static_cast<unsigned char>(s.code);
    }
  }
}

template <int LOADS, bool GROUPED>
hipError_t Launch(const MxQuantArgs& args, int64_t items, hipStream_t stream) {
  const int64_t groups = (items + kThreads * LOADS - 1) / (kThreads * LOADS);
  if (groups > 0x7fffffff) return hipErrorInvalidValue;
  hipLaunchKernelGGL((MxQuantKernel<LOADS, GROUPED>), dim3(static_cast<unsigned>(groups)), dim3(kThreads), 0, stream, args);
  return hipGetLastError();
}

}  // namespace

hipError_t PrepareMxQuantKernels() {
  hipFuncAttributes attributes;  // (no attribute to set: the calls only load the kernels onto the current device)
  const void* kernels[] = {reinterpret_cast<const void*>(&MxQuantKernel<1, false>), reinterpret_cast<const void*>(&MxQuantKernel<2, false>),
                           reinterpret_cast<const void*>(&MxQuantKernel<1, true>), reinterpret_cast<const void*>(&MxQuantKernel<2, true>)};
  for (const void* kernel : kernels) {
    if (hipError_t e = hipFuncGetAttributes(&attributes, kernel); e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t LaunchMxQuant(const MxQuantArgs& args, hipStream_t stream) {
  if (args.rows <= 0 || args.cols <= 0) return hipSuccess;
  const int64_t items = args.rows * (args.cols >> 3);
  // One item per thread while every thread has a place on the chip (256 CUs x 2048), two beyond.
  // Measured with one / two / four items per thread, rows of 64 x 512 values: 7 rows 1.95 / 2.43 / -
  // us, 100 rows 3.5 / 3.8 / 5.1, 300 rows 7.7 / 7.6 / 7.4, 1000 rows 20.3 / 18.5 / 18.5, 4096 rows
  // 74.4 / 63.6 / 65.4.
  constexpr int64_t kResidentThreads = 256 * 2048;
  if (args.group_rows > 0) {
    if (args.rows > 0xffffffffll) return hipErrorInvalidValue;
    return items <= kResidentThreads ? Launch<1, true>(args, items, stream) : Launch<2, true>(args, items, stream);
  }
  return items <= kResidentThreads ? Launch<1, false>(args, items, stream) : Launch<2, false>(args, items, stream);
}

}  // namespace mlakv
