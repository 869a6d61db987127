// aux_kernels.hip — standalone ops of the path: the mask applier and the draft map.
#include "kernels.hpp"

namespace strim {

// maskLogits (Sources/StrimCore/TokenMask.swift:15-17): where(mask, f32(logits), -inf),
// reading the packed allow-bits directly instead of a host-expanded bool row.
__global__ __launch_bounds__(256) void k_mask_logits(const void* logits, int dtype, int V,
                                                     int64_t row_stride, const uint32_t* mask,
                                                     int64_t mask_stride, float* out) {
  const int r = blockIdx.y;
  const int i0 = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (i0 >= V) return;
  uint32_t bits = 0xFu;
  if (mask) bits = (mask[(int64_t)r * mask_stride + (i0 >> 5)] >> (i0 & 31)) & 0xFu;
  for (int e = 0; e < 4 && i0 + e < V; ++e) {
    const int64_t src = (int64_t)r * row_stride + i0 + e;
    const float x = dtype == STRIM_DTYPE_BF16 ? bf16_to_f32(((const uint16_t*)logits)[src])
                                              : ((const float*)logits)[src];
    out[(int64_t)r * V + i0 + e] = ((bits >> e) & 1u) ? x : -INFINITY;
  }
}

// MTP.nextTokenIndex (Sources/StrimCore/MTP.swift:104-111): argMax over the truncated
// draft vocab (first max), then the draft->full index table.
//
// One workgroup per row: a row is at most a few hundred KB, so its time is the memory round
// trip and the reduction, and a merge across workgroups would cost a second launch. T
// threads with the 16-byte loads of N tokens each in flight (a batch): 1,024 threads of 32
// tokens take a 32,768-token row of either dtype in one (R = 4, bf16: 4.0 us against 27.7
// with 256 threads of 2-byte loads, one in flight). Rows of up to DA_SMALL tokens, and past
// DA_ROWS rows those of up to 4 DA_SMALL, take 256 threads of 8: a short row has no work for
// more, and many rows share the CUs (us, bf16, 1,024 threads against 256: R = 4, Vd = 1,001
// unaligned 4.7 and 2.8, 4,096 3.2 and 3.1, 16,384 3.6 and 4.8; R = 4,096, Vd = 4,096 20.6 and
// 8.0, 16,384 28.2 and 22.6).
// VEC: rows 16-byte aligned; other rows load token by token, in batches as wide.
constexpr int DA_SMALL = 4096, DA_ROWS = 512;
template <bool BF16, bool VEC, int T, int N>
__global__ __launch_bounds__(T) void k_draft_argmax(const void* logits, int Vd,
                                                    int64_t row_stride, const int32_t* table,
                                                    int32_t* out) {
  constexpr int DA_T = T, DA_N = N;
  __shared__ float s_v[DA_T / WAVE];
  __shared__ int s_i[DA_T / WAVE];
  const int r = blockIdx.x, t = threadIdx.x, lane = t & (WAVE - 1), w = wave_id();
  const uint16_t* xb = (const uint16_t*)logits + (int64_t)r * row_stride;
  const float* xf = (const float*)logits + (int64_t)r * row_stride;
  auto scalar = [&](int i) { return BF16 ? bf16_to_f32(xb[i]) : xf[i]; };
  constexpr int E = BF16 ? 8 : 4, U = DA_N / E;  // tokens a load, loads a batch
  float bv = -INFINITY;
  int bi = -1;
  // (a thread's ids rise: a strict compare keeps the first of equal values; NaN never wins)
  auto take = [&](float x, int i) {
    const bool up = x > bv;
    bv = up ? x : bv;
    bi = up ? i : bi;
  };
  for (int i0 = 0; i0 < Vd; i0 += DA_T * DA_N) {
    if constexpr (VEC) {
      // load u of thread t: tokens i0 + (u DA_T + t) E ..; a load that crosses the row end
      // rereads the row's start and is dropped (the row's last Vd % E tokens: below)
      uint4 q[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = i0 + (u * DA_T + t) * E;
        const int ic = i + E <= Vd ? i : 0;
        q[u] = Vd < E ? uint4{0, 0, 0, 0} : BF16 ? *(const uint4*)(xb + ic) : *(const uint4*)(xf + ic);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = i0 + (u * DA_T + t) * E;
        if (i + E > Vd) continue;
        const uint32_t wd[4] = {q[u].x, q[u].y, q[u].z, q[u].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (BF16) {
            take(__uint_as_float(wd[e] << 16), i + 2 * e);
            take(__uint_as_float(wd[e] & 0xFFFF0000u), i + 2 * e + 1);
          } else {
            take(__uint_as_float(wd[e]), i + e);
          }
        }
      }
    } else {
      float x[DA_N];
#pragma unroll
      for (int u = 0; u < DA_N; ++u) {
        const int i = i0 + u * DA_T + t;
        x[u] = scalar(i < Vd ? i : 0);
      }
#pragma unroll
      for (int u = 0; u < DA_N; ++u) {
        const int i = i0 + u * DA_T + t;
        if (i < Vd) take(x[u], i);
      }
    }
  }
  if (VEC && t < Vd % E) {
    const int i = Vd / E * E + t;
    const float x = scalar(i);
    if (x > bv) take(x, i);
  }
  auto block_best = [&]() {
    wave_argmax(bv, bi);
    if (lane == 0) {
      s_v[w] = bv;
      s_i[w] = bi;
    }
    __syncthreads();
    bv = lane < DA_T / WAVE ? s_v[lane] : -INFINITY;
    bi = lane < DA_T / WAVE ? s_i[lane] : -1;
    wave_argmax(bv, bi);
  };
  block_best();
  if (bi < 0) {
    // no value above -inf: the first that is not NaN, else index 0 (argMax over all -inf)
    __syncthreads();
    for (int i = t; i < Vd && bi < 0; i += DA_T)
      if (!isnan(scalar(i))) bi = i;
    block_best();
  }
  if (t == 0) {
    const int am = bi < 0 ? 0 : bi;
    out[r] = table ? table[am] : am;
  }
}

hipError_t launch_draft_argmax(const void* logits, bool bf16, bool vec, int R, int Vd,
                               int64_t row_stride, const int32_t* table, int32_t* out,
                               hipStream_t st) {
  const bool small = Vd <= DA_SMALL || (R > DA_ROWS && Vd <= 4 * DA_SMALL);
#define STRIM_DA(B_, V_, T_, N_)                                                              \
  hipLaunchKernelGGL((k_draft_argmax<B_, V_, T_, N_>), dim3((unsigned)R), dim3(T_), 0, st,    \
                     logits, Vd, row_stride, table, out)
#define STRIM_DA_(B_, V_)                \
  do {                                   \
    if (small) STRIM_DA(B_, V_, 256, 8); \
    else STRIM_DA(B_, V_, 1024, 32);     \
  } while (0)
  if (bf16 && vec) STRIM_DA_(true, true);
  else if (bf16) STRIM_DA_(true, false);
  else if (vec) STRIM_DA_(false, true);
  else STRIM_DA_(false, false);
#undef STRIM_DA_
#undef STRIM_DA
  return hipGetLastError();
}

}  // namespace strim
