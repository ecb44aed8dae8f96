// The reference's packed rows [T, K + 4] (e4m3 codes, then the row's fp32 dequant scale) -> what the
// GEMM reads: codes [T, K], neutral e8m0 block scales [T, K/32] and the row scales [T], in one pass.
//
// Bound by HBM: K bytes in and K * 33/32 out per row. The packed rows are 4-byte aligned only (K + 4 bytes
// apart), the codes 16-byte aligned: one wave per row reads 16 bytes per lane with 4-byte aligned
// loads, four of them in flight, and writes whole 1 KiB runs. As three torch copies and a fill
// (a strided copy each for codes and scales) it took 24 us at 3600 rows of 5120 and 115 at 32760.
#include "wanmi_common.h"

namespace wanmi {

typedef uint32_t u32x4_dword __attribute__((ext_vector_type(4), aligned(4)));

struct RowUnpackArgs {
  const uint8_t* x;  // [T] rows of K + 4 bytes, ld bytes apart
  int64_t T, K, ld;
  uint8_t* codes;      // [T, K]
  uint8_t* scales;     // [T, K/32]
  float* row_scale;    // [T]
};

constexpr uint32_t kNeutralScale = 127;  // 2^0

__global__ __launch_bounds__(256) void row_unpack_kernel(RowUnpackArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= a.T) return;
  const uint8_t* src = a.x + t * a.ld;
  uint8_t* dst = a.codes + t * a.K;
  const int chunks = (int)(a.K / 16);
  for (int c0 = 0; c0 < chunks; c0 += 256) {
    u32x4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = c0 + 64 * i + lane;
      if (c < chunks) v[i] = *reinterpret_cast<const u32x4_dword*>(src + 16 * (int64_t)c);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = c0 + 64 * i + lane;
      if (c < chunks) *reinterpret_cast<u32x4*>(dst + 16 * (int64_t)c) = v[i];
    }
  }
  const int blocks = (int)(a.K / 32);
  uint8_t* sc = a.scales + t * blocks;
  if (blocks % 4 == 0) {
    for (int i = lane; i < blocks / 4; i += 64) reinterpret_cast<uint32_t*>(sc)[i] = kNeutralScale * 0x01010101u;
  } else {
    for (int i = lane; i < blocks; i += 64) sc[i] = (uint8_t)kNeutralScale;
  }
  if (lane == 0) a.row_scale[t] = *reinterpret_cast<const float*>(src + a.K);
}

}  // namespace wanmi

extern "C" int wanmi_row_unpack(const void* packed, int64_t T, int64_t K, int64_t ld, void* codes, uint8_t* scales,
                                float* row_scale, void* stream) {
  using namespace wanmi;
  clear_error();
  WANMI_REQUIRE(T >= 0 && K > 0 && K % 32 == 0 && K < (1LL << 31) && ld >= K + 4, WANMI_ERR_ARG,
                "wanmi_row_unpack: need K a positive multiple of 32 and ld >= K + 4 (T=%lld K=%lld ld=%lld)", (long long)T,
                (long long)K, (long long)ld);
  if (T == 0) return WANMI_OK;
  WANMI_REQUIRE(packed && codes && scales && row_scale, WANMI_ERR_ARG, "wanmi_row_unpack: null pointer");
  WANMI_REQUIRE(((uintptr_t)packed % 4) == 0 && ld % 4 == 0 && ((uintptr_t)codes % 16) == 0 &&
                    ((uintptr_t)scales % 4) == 0 && ((uintptr_t)row_scale % 4) == 0,
                WANMI_ERR_ARG, "wanmi_row_unpack: rows, scales and row_scale must be 4-byte, codes 16-byte aligned");
  const int64_t groups = (T + 3) / 4;
  WANMI_REQUIRE(groups < (1LL << 31), WANMI_ERR_ARG, "wanmi_row_unpack: too many rows");
  RowUnpackArgs a;
  a.x = static_cast<const uint8_t*>(packed);
  a.T = T;
  a.K = K;
  a.ld = ld;
  a.codes = static_cast<uint8_t*>(codes);
  a.scales = scales;
  a.row_scale = row_scale;
  hipLaunchKernelGGL(row_unpack_kernel, dim3((unsigned)groups), dim3(256), 0, (hipStream_t)stream, a);
  return check_launch("wanmi_row_unpack");
}
