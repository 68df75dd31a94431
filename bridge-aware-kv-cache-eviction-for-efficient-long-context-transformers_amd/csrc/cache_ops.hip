// The evicting caches' per-step work: a layer's new K and V rows appended to
// its buffers (cab_kv_append), and attention weights summed into the running
// importance totals (cab_key_sums). Decode steps run these on a few KB, so
// each is one launch; the prefill's are HBM-bound. A pass of 8 layers x (a
// prefill of 4500 rows + 12 tokens), 8 heads, D = 128, bf16: 146 launches and
// 557 us of kernels (in the profiler), against 320 and 1133 us as torch copies,
// zero fills, sums and concatenations; 2465 -> 2007 us with the host's part.
#include "cab_internal.h"

namespace cab {
namespace {

struct AppendArgs {
  const char* src[2];  // K, V: row 0 of the new rows
  char* dst[2];        // K, V: where the first new row goes
  int64_t ss[2][4];    // source strides in bytes: b, h, row, element
  int64_t ds[3];       // destination strides in bytes: b, h, row (K and V alike)
  uint32_t H, n, units;  // units: copies of U bytes per row
  uint64_t total;      // B * H * n * units
};

// U bytes per thread and step; blockIdx.y: K or V. U = 16 when rows are
// contiguous and 16-byte aligned on both sides, else the element size.
template <typename U>
__global__ __launch_bounds__(256) void kv_append_kernel(AppendArgs a) {
  const int t = blockIdx.y;
  const char* src = a.src[t];
  char* dst = a.dst[t];
  const int64_t s0 = a.ss[t][0], s1 = a.ss[t][1], s2 = a.ss[t][2], s3 = a.ss[t][3];
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x; i < a.total;
       i += static_cast<uint64_t>(gridDim.x) * 256) {
    // (total < 2^32: the host takes larger appends in parts)
    const uint32_t x = static_cast<uint32_t>(i);
    const uint32_t row = x / a.units, u = x - row * a.units;
    const uint32_t bh = row / a.n, r = row - bh * a.n;
    const uint32_t b = bh / a.H, h = bh - b * a.H;
    *reinterpret_cast<U*>(dst + b * a.ds[0] + h * a.ds[1] + r * a.ds[2] +
                          static_cast<int64_t>(u) * sizeof(U)) =
        *reinterpret_cast<const U*>(src + b * s0 + h * s1 + r * s2 + u * s3);
  }
}

struct SumArgs {
  const void* a;
  int64_t st[4];  // elements: b, h, query, key
  uint32_t H, Nq, rows;
  int32_t Nk;
  const float* old;  // may be out
  int32_t n_old, n_out;
  float* out;
};

// One workgroup of 16 waves per 64 keys: wave w sums the rows (b, h, query)
// w, w + 16, .., eight at a time, as trees of additions; so are the waves' sums.
// 16-bit weights: the sum is rounded to their type before it is added, as a
// torch sum of them is.
constexpr int SUM_WAVES = 16;
template <typename T>
__global__ __launch_bounds__(64 * SUM_WAVES) void key_sums_kernel(SumArgs a) {
  __shared__ float part[SUM_WAVES][64];
  const int lane = lane_id(), w = threadIdx.x >> 6;
  const int key = blockIdx.x * 64 + lane;
  float sum = 0.f;
  if (key < a.Nk) {
    const int64_t at = key * a.st[3];
    // Eight rows are loaded before any is added.
    constexpr int U = 8;
    for (uint32_t r0 = w; r0 < a.rows; r0 += U * SUM_WAVES) {
      float x[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t r = r0 + u * SUM_WAVES;
        x[u] = 0.f;
        if (r < a.rows) {
          const uint32_t bh = r / a.Nq, q = r - bh * a.Nq;
          const uint32_t b = bh / a.H, h = bh - b * a.H;
          const int64_t off = b * a.st[0] + h * a.st[1] + q * a.st[2] + at;
          if constexpr (std::is_same<T, float>::value)
            x[u] = static_cast<const float*>(a.a)[off];
          else if constexpr (std::is_same<T, bf16_t>::value)
            x[u] = bf16_to_f32(static_cast<const uint16_t*>(a.a)[off]);
          else
            x[u] = f16_to_f32(static_cast<const uint16_t*>(a.a)[off]);
        }
      }
      sum += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
    }
  }
  part[w][lane] = sum;
  __syncthreads();
  if (w != 0 || key >= a.n_out) return;
  float y[SUM_WAVES];
#pragma unroll
  for (int i = 0; i < SUM_WAVES; ++i) y[i] = part[i][lane];
#pragma unroll
  for (int n = SUM_WAVES / 2; n >= 1; n >>= 1)
#pragma unroll
    for (int i = 0; i < n; ++i) y[i] = y[2 * i] + y[2 * i + 1];
  sum = y[0];
  if constexpr (std::is_same<T, bf16_t>::value)
    sum = bf16_to_f32(f32_to_bf16(sum));
  else if constexpr (std::is_same<T, f16_t>::value)
    sum = f16_to_f32(f32_to_f16(sum));
  a.out[key] = (key < a.n_old ? a.old[key] : 0.f) + sum;
}

}  // namespace
}  // namespace cab

using namespace cab;

extern "C" cab_status_t cab_kv_append(const void* k, const void* v, void* k_dst, void* v_dst,
                                      int32_t element_bytes, int64_t B, int64_t H, int64_t n,
                                      int64_t D, const int64_t k_strides[4],
                                      const int64_t v_strides[4], const int64_t dst_strides[4],
                                      int64_t dst_row, void* stream) {
  const char* fn = "cab_kv_append";
  clear_error();
  CAB_REQUIRE(element_bytes == 2 || element_bytes == 4, CAB_EDTYPE,
              "%s: element size %d unsupported (2 or 4)", fn, (int)element_bytes);
  CAB_REQUIRE(B >= 0 && H >= 0 && n >= 0 && D >= 0 && dst_row >= 0, CAB_ESHAPE,
              "%s: negative size", fn);
  if (B == 0 || H == 0 || n == 0 || D == 0) return CAB_OK;
  CAB_REQUIRE(k && v && k_dst && v_dst && k_strides && v_strides && dst_strides, CAB_EINVAL,
              "%s: null argument", fn);
  CAB_REQUIRE(dst_strides[3] == 1, CAB_ESHAPE, "%s: the buffers' last-dim stride must be 1", fn);
  const int64_t es = element_bytes;
  AppendArgs a;
  const void* src[2] = {k, v};
  void* dst[2] = {k_dst, v_dst};
  const int64_t* st[2] = {k_strides, v_strides};
  bool wide = D * es % 16 == 0;
  for (int t = 0; t < 2; ++t) {
    CAB_REQUIRE(reinterpret_cast<uintptr_t>(src[t]) % es == 0 &&
                    reinterpret_cast<uintptr_t>(dst[t]) % es == 0,
                CAB_ESHAPE, "%s: pointers not aligned to their elements", fn);
    a.src[t] = static_cast<const char*>(src[t]);
    a.dst[t] = static_cast<char*>(dst[t]) + dst_row * dst_strides[2] * es;
    wide = wide && st[t][3] == 1 && reinterpret_cast<uintptr_t>(a.src[t]) % 16 == 0 &&
           reinterpret_cast<uintptr_t>(a.dst[t]) % 16 == 0;
    for (int d = 0; d < 4; ++d) a.ss[t][d] = st[t][d] * es;
    for (int d = 0; d < 3; ++d) wide = wide && a.ss[t][d] % 16 == 0;
  }
  for (int d = 0; d < 3; ++d) {
    a.ds[d] = dst_strides[d] * es;
    wide = wide && a.ds[d] % 16 == 0;
  }
  const int64_t units = wide ? D * es / 16 : D;
  if (wide) a.ss[0][3] = a.ss[1][3] = 16;
  // 32-bit indexes: at most 2^31 units a launch, in whole parts of the rows.
  CAB_REQUIRE(B <= INT32_MAX / H && B * H <= INT32_MAX / units, CAB_ESHAPE, "%s: B * H * D too large", fn);
  const int64_t most = INT32_MAX / (B * H * units);
  hipStream_t s = static_cast<hipStream_t>(stream);
  for (int64_t r0 = 0; r0 < n; r0 += most) {
    const int64_t m = n - r0 < most ? n - r0 : most;
    a.H = static_cast<uint32_t>(H);
    a.n = static_cast<uint32_t>(m);
    a.units = static_cast<uint32_t>(units);
    a.total = static_cast<uint64_t>(B * H * m * units);
    const int64_t blocks = ceil_div(static_cast<int64_t>(a.total), 256);
    const dim3 grid(static_cast<unsigned>(blocks < 4096 ? blocks : 4096), 2);
    if (wide)
      kv_append_kernel<u32x4><<<grid, 256, 0, s>>>(a);
    else if (es == 4)
      kv_append_kernel<uint32_t><<<grid, 256, 0, s>>>(a);
    else
      kv_append_kernel<uint16_t><<<grid, 256, 0, s>>>(a);
    const cab_status_t r = launch_status(fn);
    if (r != CAB_OK) return r;
    for (int t = 0; t < 2; ++t) {
      a.src[t] += m * a.ss[t][2];
      a.dst[t] += m * a.ds[2];
    }
  }
  return CAB_OK;
}

extern "C" cab_status_t cab_key_sums(const void* attention, cab_dtype_t dtype, int64_t B, int64_t H,
                                     int64_t N_q, int64_t N_k, const int64_t strides[4],
                                     const float* old_sums, int64_t n_old, float* sums,
                                     void* stream) {
  const char* fn = "cab_key_sums";
  clear_error();
  CAB_REQUIRE(valid_dtype(dtype), CAB_EDTYPE, "%s: unknown dtype %d", fn, static_cast<int>(dtype));
  CAB_REQUIRE(B >= 1 && H >= 1 && N_q >= 1 && N_k >= 1 && n_old >= 0, CAB_ESHAPE, "%s: bad shape", fn);
  CAB_REQUIRE(B <= INT32_MAX / H && N_q <= INT32_MAX / (B * H) && N_k <= INT32_MAX - 64 &&
                  n_old <= INT32_MAX - 64,
              CAB_ESHAPE, "%s: problem too large", fn);
  CAB_REQUIRE(attention && sums && strides && (n_old == 0 || old_sums), CAB_EINVAL,
              "%s: null argument", fn);
  SumArgs a;
  a.a = attention;
  for (int d = 0; d < 4; ++d) a.st[d] = strides[d];
  a.H = static_cast<uint32_t>(H);
  a.Nq = static_cast<uint32_t>(N_q);
  a.rows = static_cast<uint32_t>(B * H * N_q);
  a.Nk = static_cast<int32_t>(N_k);
  a.old = old_sums;
  a.n_old = static_cast<int32_t>(n_old);
  a.n_out = a.Nk;
  a.out = sums;
  const unsigned grid = static_cast<unsigned>(ceil_div(a.n_out, 64));
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case CAB_F32: key_sums_kernel<float><<<grid, 64 * SUM_WAVES, 0, s>>>(a); break;
    case CAB_BF16: key_sums_kernel<bf16_t><<<grid, 64 * SUM_WAVES, 0, s>>>(a); break;
    default: key_sums_kernel<f16_t><<<grid, 64 * SUM_WAVES, 0, s>>>(a); break;
  }
  return launch_status(fn);
}
