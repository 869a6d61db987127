// head_kernels.hip — the producer of the logits the path reads: the decode step's final
// RMSNorm and lm_head linear (QwenModel.swift:202-212; Weights.swift:244-255,270-273), for
// dense bf16 weights, on MFMA, writing the bf16 logits in the layout strim_sample takes.
//
// k_head_norm: one workgroup per row, xn = bf16(w * bf16(x * inv)) with
//   inv = 1 / sqrt(mean(x^2) + eps), the squares summed in double.
// k_head_split (most calls of up to 16 rows, and more rows on small vocabularies),
// k_head_gemv (the others; launch_head has the lines):
//   logits[b][v] = bf16(sum_k xn[b][k] W[v][k]) with float accumulation. The weight matrix
//   is read exactly once per call whatever the batch, which is the MFMA's N side (16 rows
//   per tile, up to four tiles). k_head_split: a workgroup owns 32 or 64 vocabulary rows and
//   its waves split K; the batch operand comes from the L2-resident xn. k_head_gemv: a
//   workgroup owns 128 vocabulary rows, each wave two 16-row tiles over the whole of K,
//   and the workgroup stages xn in LDS. Both add a logit's products in one order (head_segs).
//   For a greedy pick (strim_head_greedy) its epilogue also writes each batch row's first
//   maximum over the workgroup's logits (as bf16 values, as the sampler reads them),
//   and the logits may be left unwritten.
// k_head_pick: one workgroup per batch row merges the rows' tile maxima into the first
//   maximum of the row: the greedy token, with the sampler's statuses (a NaN or +inf logit:
//   STRIM_ENONFINITE; every logit -inf: STRIM_EEMPTY).
//
// MFMA operand layout (v_mfma_f32_16x16x32_bf16; checked on the device): lane l holds
// A[l % 16][8 (l / 16) + i] and B[8 (l / 16) + i][l % 16] for i < 8, and C[4 (l / 16) + i]
// [l % 16] for i < 4. A step of 128 elements of K is four MFMAs; MFMA q takes elements
// 32 q + 8 (l / 16) + i of the weight row and of the xn row, so each wave-wide load reads
// 64 contiguous bytes of each of 16 rows.
#include "kernels.hpp"

namespace strim {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int HN_T = 1024;              // k_head_norm threads
constexpr int HG_W = 4;                 // k_head_gemv waves per workgroup
constexpr int HG_MT = 2;                // 16-row vocabulary tiles per wave
constexpr int HG_KS = 128;              // K elements per step (four MFMAs of K 32)

// Every kernel adds a logit's products in one order, which K alone fixes: K's n steps fall
// into head_segs(K) segments, segment i the steps [i n / S, (i + 1) n / S); each segment is
// one accumulator chain from zero, and the segments' sums are added in order. So a row's
// logits are the same bits whatever the batch and the vocabulary it is computed with.
constexpr int head_segs(int K) { return K >= 4096 ? 8 : 4; }

// Round to nearest even; NaN stays a quiet NaN.
__device__ __forceinline__ uint16_t head_bf16(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7FFFFFFFu) > 0x7F800000u) return (uint16_t)((u >> 16) | 0x0040u);
  return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

__global__ __launch_bounds__(HN_T) void k_head_norm(const uint16_t* x, int64_t x_stride, int K,
                                                    const uint16_t* w, float eps,
                                                    uint16_t* xn) {
  __shared__ double s_d[HN_T / WAVE];
  const int b = blockIdx.x, t = threadIdx.x;
  const uint16_t* xr = x + (int64_t)b * x_stride;
  double ss = 0.0;
  // A row's time is its chain of round trips: the first 8 HN_T elements' row and weight
  // pieces (all of them up to K = 8,192) are requested together and held, so the
  // normalisation after the sum waits for no second trip (K = 5,120: 6.0 -> 4.6 us; 256
  // threads read the row twice).
  const int k0 = 8 * t < K ? 8 * t : 0;
  const uint4 q0 = *(const uint4*)(xr + k0), g0 = *(const uint4*)(w + k0);
  for (int k = 8 * t; k < K; k += 8 * HN_T) {
    const uint4 q = k == k0 ? q0 : *(const uint4*)(xr + k);
    const uint32_t wd[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float lo = __uint_as_float(wd[e] << 16), hi = __uint_as_float(wd[e] & 0xFFFF0000u);
      ss += (double)lo * (double)lo + (double)hi * (double)hi;
    }
  }
  ss = wave_sum(ss);
  if ((t & (WAVE - 1)) == 0) s_d[t / WAVE] = ss;
  __syncthreads();
  double tot = 0.0;
#pragma unroll
  for (int q = 0; q < HN_T / WAVE; ++q) tot += s_d[q];
  const float inv = 1.0f / sqrtf((float)(tot / (double)K) + eps);
  for (int k = 8 * t; k < K; k += 8 * HN_T) {
    const uint4 q = k == k0 ? q0 : *(const uint4*)(xr + k);
    const uint4 g = k == k0 ? g0 : *(const uint4*)(w + k);
    const uint32_t xd[4] = {q.x, q.y, q.z, q.w}, gd[4] = {g.x, g.y, g.z, g.w};
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t r = 0u;
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        const float xv = __uint_as_float(hf ? (xd[e] & 0xFFFF0000u) : (xd[e] << 16));
        const float gv = __uint_as_float(hf ? (gd[e] & 0xFFFF0000u) : (gd[e] << 16));
        const float y = bf16_to_f32(head_bf16(xv * inv));
        r |= (uint32_t)head_bf16(gv * y) << (16 * hf);
      }
      o[e] = r;
    }
    *(uint4*)(xn + (int64_t)b * K + k) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

// The larger of two (value, id) pairs, the smaller id on equal values (NaN never taken).
__device__ __forceinline__ void hb_take(float& v, int& i, float v2, int i2) {
  if (v2 > v || (v2 == v && i2 < i)) {
    v = v2;
    i = i2;
  }
}

// Four logits of one batch row, vocabulary ids vb .. vb + 3 (those below V).
template <bool VO>
__device__ __forceinline__ void head_store4(uint16_t* dst, const uint16_t* o, int vb, int V) {
  if (VO && vb + 3 < V) {
    *(uint2*)dst = make_uint2((uint32_t)o[0] | ((uint32_t)o[1] << 16),
                              (uint32_t)o[2] | ((uint32_t)o[3] << 16));
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (vb + i < V) dst[i] = o[i];
  }
}

// NT: 16-row batch tiles (B <= 16 NT). VO: 8-byte logit stores (rows 4-element aligned).
// TB: write the tile maxima to tbest[n][blockIdx.x] = {value bits (NaN: the tile holds a
// NaN or +inf), id}; out NULL: no logits stored. MT: 16-row vocabulary tiles per wave; NW:
// waves per workgroup.
template <int NT, bool VO, bool TB, int MT, int NW>
__global__ __launch_bounds__(NW* WAVE, NT == 2 ? 4 : 1) void k_head_gemv(const uint16_t* xn, int64_t xn_stride,
                                                          int B, int K, const uint16_t* W,
                                                          int64_t w_stride, int V,
                                                          uint16_t* out, int64_t out_stride,
                                                          uint2* tbest) {
  const int lane = threadIdx.x & (WAVE - 1), wv = wave_id();
  const int h = lane >> 4, r16 = lane & 15;
  const int v0 = blockIdx.x * (NW * MT * 16) + wv * (MT * 16);
  // rows past V or B read a clamped row; their results are not stored
  const uint16_t* arow[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int v = min(v0 + mt * 16 + r16, V - 1);
    arow[mt] = W + (int64_t)v * w_stride + 8 * h;
  }
  // the current segment's sums, and the finished segments': two batch tiles keep those in
  // LDS (each thread its own) and four waves a SIMD (B = 24, V = 151,936, K = 5,120: 287.7 us,
  // 291.1 with the registers at three waves, 297.8 with them at four; one chain over the whole
  // of K, without the segments, 288.3)
  constexpr bool LT = NT == 2;
  __shared__ f32x4_t s_tot[LT ? MT * NT : 1][LT ? NW * WAVE : 1];
  f32x4_t acc[MT][NT], tot[LT ? 1 : MT][LT ? 1 : NT];
  auto total = [&](int mt, int nt) -> f32x4_t& {
    if constexpr (LT) return s_tot[mt * NT + nt][threadIdx.x];
    else return tot[mt][nt];
  };
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = total(mt, nt) = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // two register buffers: the next step's loads are in flight while this step multiplies
  uint4 a[2][MT][4];
  auto loada = [&](int buf, int kb) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int q = 0; q < 4; ++q) a[buf][mt][q] = *(const uint4*)(arow[mt] + kb + 32 * q);
  };
  // K is a multiple of 2 steps (the host checks), so every load and multiply is
  // unconditional (the last prefetch reloads the last step and is not used), and the
  // scheduling barriers keep each buffer's loads issued before the other buffer's
  // multiplies: left alone, the compiler sinks the loads next to their use
  const int nsteps = K / HG_KS, segs = head_segs(K);
  int seg = 1, seg_end = nsteps / segs;
  // after `done` steps: a finished segment's sums join the total (a segment may be empty)
  auto end_step = [&](int done) {
    if (done < seg_end || done == nsteps) return;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        total(mt, nt) += acc[mt][nt];
        acc[mt][nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    do {
      ++seg;
      seg_end = seg * nsteps / segs;
    } while (seg_end <= done);
  };
  // Several batch tiles: every wave needs the same 16 NT rows of xn at each step, so
  // the workgroup stages them in LDS once (double-buffered, rows padded by 16 bytes so
  // the 16 rows a wave reads fall in different banks) instead of each wave reading
  // them from L2 (four times the bytes: that bound B = 64 at 2.7 TB/s). Thread t
  // carries NT 16-byte pieces of the next step's slice while this step multiplies.
  constexpr int XR = 16 * NT, XW = HG_KS + 8;  // rows, padded row length (bf16)
  __shared__ __attribute__((aligned(16))) uint16_t s_x[2][XR][XW];
  struct Slice {
    uint4 v[NT];
  };
  auto xload = [&](int kb) -> Slice {
    Slice xr;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int e = (int)threadIdx.x + NW * WAVE * i;  // piece e: row e / 16, column 8 (e % 16)
      const int row = e >> 4, col = (e & 15) * 8;
      const int n = min(row, B - 1);
      xr.v[i] = *(const uint4*)(xn + (int64_t)n * xn_stride + kb + col);
    }
    return xr;
  };
  auto xstore = [&](int buf, const Slice& xr) {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int e = (int)threadIdx.x + NW * WAVE * i;
      *(uint4*)&s_x[buf][e >> 4][(e & 15) * 8] = xr.v[i];
    }
  };
  // the multiplies of one step from LDS buffer buf, the B operand read one K slice (q)
  // at a time next to its MFMAs: NT registers of it live instead of 4 NT
  auto mma_lds = [&](int buf, int abuf) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint4 bx[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        bx[nt] = *(const uint4*)&s_x[buf][nt * 16 + r16][32 * q + 8 * h];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8_t, a[abuf][mt][q]), __builtin_bit_cast(bf16x8_t, bx[nt]),
              acc[mt][nt], 0, 0, 0);
    }
  };
  static_assert(NT * NW * WAVE * 8 == XR * HG_KS, "one step's slice: NT pieces a thread");
  // The barrier waits for the LDS stores alone: __syncthreads' fence would also wait
  // for the next step's weight loads, the prefetch this loop depends on. The slice's
  // loads are issued before the weights', so its store waits for them only.
  auto sync_lds = []() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  // Unrolled by two so each register buffer has a fixed index (the host checks that K
  // is a multiple of two steps; the last prefetch reloads the last step, unused).
  xstore(0, xload(0));
  loada(0, 0);
  sync_lds();
  for (int s = 0; s < nsteps; s += 2) {
    const Slice x1 = xload((s + 1) * HG_KS);
    loada(1, (s + 1) * HG_KS);
    __builtin_amdgcn_sched_barrier(0);
    mma_lds(0, 0);
    end_step(s + 1);
    __builtin_amdgcn_sched_barrier(0);
    xstore(1, x1);
    sync_lds();
    const int s2 = min(s + 2, nsteps - 2) * HG_KS;
    const Slice x0 = xload(s2);
    loada(0, s2);
    __builtin_amdgcn_sched_barrier(0);
    mma_lds(1, 1);
    end_step(s + 2);
    __builtin_amdgcn_sched_barrier(0);
    xstore(0, x0);
    sync_lds();
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = total(mt, nt) + acc[mt][nt];
  // lane l holds rows 4 h + i of each tile for batch row nt 16 + r16
  float bv[NT];
  int bi[NT];
  bool bad[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    bv[nt] = -INFINITY;
    bi[nt] = INT_MAX;
    bad[nt] = false;
    const int n = nt * 16 + r16;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int vb = v0 + mt * 16 + 4 * h;
      uint16_t o[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = head_bf16(acc[mt][nt][i]);
      if constexpr (TB) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (vb + i < V) {
            const float f = __uint_as_float((uint32_t)o[i] << 16);
            bad[nt] = bad[nt] || !(f < INFINITY);  // NaN or +inf
            hb_take(bv[nt], bi[nt], f, vb + i);
          }
      }
      if (n >= B || out == nullptr) continue;
      uint16_t* dst = out + (int64_t)n * out_stride + vb;
      head_store4<VO>(dst, o, vb, V);
    }
  }
  if constexpr (TB) {
    // the four lanes of a batch row (h = 0..3), then the workgroup's waves
    __shared__ float s_v[NW][16 * NT];
    __shared__ int s_i[NW][16 * NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
      for (int sh = 16; sh < WAVE; sh <<= 1) {
        const float v2 = __shfl_xor(bv[nt], sh);
        const int i2 = __shfl_xor(bi[nt], sh);
        const bool b2 = __shfl_xor((int)bad[nt], sh) != 0;
        hb_take(bv[nt], bi[nt], v2, i2);
        bad[nt] = bad[nt] || b2;
      }
      if (h == 0) {
        s_v[wv][nt * 16 + r16] = bad[nt] ? __uint_as_float(0x7FC00000u) : bv[nt];
        s_i[wv][nt * 16 + r16] = bi[nt];
      }
    }
    __syncthreads();
    const int n = (int)threadIdx.x;
    if (n < B && n < 16 * NT) {
      float v = s_v[0][n];
      int i = s_i[0][n];
      bool nan = !(v == v);
#pragma unroll
      for (int q = 1; q < NW; ++q) {
        nan = nan || !(s_v[q][n] == s_v[q][n]);
        hb_take(v, i, s_v[q][n], s_i[q][n]);
      }
      tbest[(int64_t)n * gridDim.x + blockIdx.x] =
          make_uint2(__float_as_uint(nan ? __uint_as_float(0x7FC00000u) : v), (uint32_t)i);
    }
  }
}

// The same product with K split over the workgroup's waves: wave w multiplies the steps
// [w n / NW, (w + 1) n / NW) of the same MT 16-row tiles, and the partial sums are added in
// wave order through LDS (NW = head_segs(K): a wave's steps are one segment). Bound by HBM. A
// workgroup that holds 128 rows over the whole of K leaves the chip half empty at its end,
// or throughout where V / 128 is near or below the 256 CUs; 32 rows are a quarter of its
// work, and a wave does a quarter (four waves) or an eighth (eight) of what one of its four
// waves did (each wave's batch slice is read from L2 either way at one batch tile). B = 8, K = 5,120: 109.6 -> 77.8 us at
// V = 40,000 (65 at a plain read's 6.26 TB/s), 54.4 -> 21.6 at V = 8,192, 280.0 -> 272.8 at
// V = 151,936; K = 2,048, V = 151,936: 143.5 -> 109.7.
template <int NT, bool VO, bool TB, int MT, int NW>
__global__ __launch_bounds__(NW* WAVE) void k_head_split(const uint16_t* xn, int64_t xn_stride,
                                                           int B, int K, const uint16_t* W,
                                                           int64_t w_stride, int V,
                                                           uint16_t* out, int64_t out_stride,
                                                           uint2* tbest) {
  __shared__ f32x4_t s_acc[NW][MT * NT][WAVE];
  const int lane = threadIdx.x & (WAVE - 1), wv = wave_id();
  const int h = lane >> 4, r16 = lane & 15;
  const int v0 = blockIdx.x * (MT * 16);
  const int nsteps = K / HG_KS, s0 = wv * nsteps / NW, n = (wv + 1) * nsteps / NW - s0;
  // rows past V or B read a clamped row; their results are not stored
  const uint16_t* arow[MT];
  const uint16_t* brow[NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    arow[mt] = W + (int64_t)min(v0 + mt * 16 + r16, V - 1) * w_stride + 8 * h + s0 * HG_KS;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
    brow[nt] = xn + (int64_t)min(nt * 16 + r16, B - 1) * xn_stride + 8 * h + s0 * HG_KS;
  f32x4_t acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  uint4 a[2][MT][4], bq[2][NT][4];
  auto load = [&](int buf, int s) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int q = 0; q < 4; ++q) a[buf][mt][q] = *(const uint4*)(arow[mt] + s * HG_KS + 32 * q);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int q = 0; q < 4; ++q) bq[buf][nt][q] = *(const uint4*)(brow[nt] + s * HG_KS + 32 * q);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto mma = [&](int buf) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8_t, a[buf][mt][q]),
              __builtin_bit_cast(bf16x8_t, bq[buf][nt][q]), acc[mt][nt], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  // (a wave may have no step when K has fewer than NW; the last one or two steps are peeled,
  // so that no load in the loop is conditional and none is repeated)
  if (n > 0) {
    load(0, 0);
    int s = 0;
    for (; s + 2 < n; s += 2) {
      load(1, s + 1);
      mma(0);
      load(0, s + 2);
      mma(1);
    }
    if (s + 2 == n) {
      load(1, s + 1);
      mma(0);
      mma(1);
    } else {
      mma(0);
    }
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) s_acc[wv][nt * MT + mt][lane] = acc[mt][nt];
  __syncthreads();
  __shared__ float s_v[TB ? MT : 1][16 * NT];
  __shared__ int s_i[TB ? MT : 1][16 * NT];
  // tile e of wave e % NW; lane l holds rows 4 h + i of it for batch row nt 16 + r16
#pragma unroll
  for (int e0 = 0; e0 < MT * NT; e0 += NW) {
    const int e = e0 + wv;
    if (e >= MT * NT) break;
    const int mt = e % MT, nr = e / MT * 16 + r16, vb = v0 + mt * 16 + 4 * h;
    f32x4_t sum = s_acc[0][e][lane];
#pragma unroll
    for (int q = 1; q < NW; ++q) sum += s_acc[q][e][lane];
    uint16_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = head_bf16(sum[i]);
    if (nr < B && out != nullptr) head_store4<VO>(out + (int64_t)nr * out_stride + vb, o, vb, V);
    if constexpr (TB) {
      float bv = -INFINITY;
      int bi = INT_MAX;
      bool bad = false;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (vb + i < V) {
          const float f = __uint_as_float((uint32_t)o[i] << 16);
          bad = bad || !(f < INFINITY);  // NaN or +inf
          hb_take(bv, bi, f, vb + i);
        }
#pragma unroll
      for (int sh = 16; sh < WAVE; sh <<= 1) {
        const float v2 = __shfl_xor(bv, sh);
        const int i2 = __shfl_xor(bi, sh);
        bad = (__shfl_xor((int)bad, sh) != 0) || bad;
        hb_take(bv, bi, v2, i2);
      }
      if (h == 0) {
        s_v[mt][nr] = bad ? __uint_as_float(0x7FC00000u) : bv;
        s_i[mt][nr] = bi;
      }
    }
  }
  if constexpr (TB) {
    __syncthreads();
    const int nr = (int)threadIdx.x;
    if (nr < B && nr < 16 * NT) {
      float v = s_v[0][nr];
      int i = s_i[0][nr];
      bool nan = !(v == v);
#pragma unroll
      for (int q = 1; q < MT; ++q) {
        nan = nan || !(s_v[q][nr] == s_v[q][nr]);
        hb_take(v, i, s_v[q][nr], s_i[q][nr]);
      }
      tbest[(int64_t)nr * gridDim.x + blockIdx.x] =
          make_uint2(__float_as_uint(nan ? __uint_as_float(0x7FC00000u) : v), (uint32_t)i);
    }
  }
}

// One workgroup a batch row: the row's tile maxima (4,748 of 32 vocabulary rows each at
// V = 151,936) in batches of HP_U loads a thread, all in flight. The fused greedy call at
// B = 8, K = 5,120, V = 151,936 takes 286.7 us with the logits written and 277.7 without
// (292.7 and 283.7 with 256 threads and one load in flight; the producer and strim_sample
// 283.8).
constexpr int HP_T = 1024, HP_U = 8;

__global__ __launch_bounds__(HP_T) void k_head_pick(const uint2* tbest, int ntiles,
                                                     int32_t* out_ids, int32_t* out_status) {
  __shared__ float s_v[HP_T / WAVE];
  __shared__ int s_i[HP_T / WAVE], s_bad[HP_T / WAVE];
  const int n = blockIdx.x, t = threadIdx.x, lane = t & (WAVE - 1), w = wave_id();
  const uint2* row = tbest + (int64_t)n * ntiles;
  float v = -INFINITY;
  int i = INT_MAX;
  bool bad = false;
  auto merge = [&](int width) {
    for (int sh = 1; sh < width; sh <<= 1) {
      const float v2 = __shfl_xor(v, sh);
      const int i2 = __shfl_xor(i, sh);
      bad = (__shfl_xor((int)bad, sh) != 0) || bad;
      hb_take(v, i, v2, i2);
    }
  };
  for (int q0 = t; q0 < ntiles; q0 += HP_T * HP_U) {
    uint2 r[HP_U];
#pragma unroll
    for (int u = 0; u < HP_U; ++u) r[u] = row[min(q0 + u * HP_T, ntiles - 1)];
#pragma unroll
    for (int u = 0; u < HP_U; ++u) {  // (past the row: its last tile again)
      const float f = __uint_as_float(r[u].x);
      bad = bad || !(f == f);
      hb_take(v, i, f, (int)r[u].y);
    }
  }
  merge(WAVE);
  if (lane == 0) {
    s_v[w] = v;
    s_i[w] = i;
    s_bad[w] = bad ? 1 : 0;
  }
  __syncthreads();
  if (w == 0) {
    const int q = lane & (HP_T / WAVE - 1);
    v = s_v[q];
    i = s_i[q];
    bad = s_bad[q] != 0;
    merge(HP_T / WAVE);
    if (t == 0) {
      const int st = bad ? STRIM_ENONFINITE : (v > -INFINITY ? STRIM_OK : STRIM_EEMPTY);
      out_ids[n] = st == STRIM_OK ? i : -1;
      if (out_status) out_status[n] = st;
    }
  }
}

hipError_t launch_head(const void* hidden, int64_t hidden_stride, int B, int K,
                       const void* norm_w, float eps, void* xn, const void* W, int64_t w_stride,
                       int V, void* out, int64_t out_stride, bool vo, hipStream_t st,
                       uint2* tbest, int32_t* out_ids, int32_t* out_status) {
  const uint16_t* src = (const uint16_t*)hidden;
  int64_t src_stride = hidden_stride;
  if (norm_w) {
    hipLaunchKernelGGL(k_head_norm, dim3((unsigned)B), dim3(HN_T), 0, st, (const uint16_t*)hidden,
                       hidden_stride, K, (const uint16_t*)norm_w, eps, (uint16_t*)xn);
    src = (const uint16_t*)xn;
    src_stride = K;
  }
  // One batch tile: K split over eight waves where it has eight segments (head_segs), else
  // four. 32 vocabulary rows a workgroup; at K from 4,096, two forms read xn less often,
  // which counts where its tile's rows are distinct: 64 rows a workgroup, and the staged
  // kernel (its build for two tiles). Both take their time in whole rounds over the 256
  // CUs, of 16,384 and 32,768 rows, so they are for vocabularies that nearly fill their
  // last round, the more nearly the fewer rows there are. K = 5,120, us for 32 rows, 64
  // rows, staged: V = 151,936 (rounds 93 % full) B = 10 286 289 279, B = 16 315 302 284;
  // V = 65,536 (full) B = 10 125.0 123.0 118.1; V = 80,000 (98 and 81 %) B = 12 161 153
  // 164; V = 100,000 (87 and 76 %) B = 12 201 206 215, B = 16 213 210 217. Where K is a
  // multiple of 2,048 the staged kernel's rows meet in few memory channels (K = 6,144,
  // V = 131,072, B = 16: 299 300 325; K = 8,192, V = 128,256: 432 385 451).
  // More tiles: the staged slice of xn is worth more than the split, until its 128-row
  // workgroups leave most CUs idle (its time hardly falls below V = 20,000, the split's is
  // in proportion to V. K = 5,120, V = 8,192: B = 24 50.4 -> 26.5 us, B = 64 59.1 -> 37.8;
  // V = 20,000: B = 24 56.1 against 62.0, B = 64 65 against 97; K = 3,584, V = 10,672:
  // B = 24 36.9 -> 30.7, B = 64 42.9 against 47.1).
  const bool deep = head_segs(K) == 8;
  auto fills = [&](int unit) {  // the rounds of `unit` rows are (103 - B) % full or more
    const int64_t rounds = ((int64_t)V + unit - 1) / unit;
    return 100 * (int64_t)V >= (103 - B) * unit * rounds;
  };
  const bool wide1 = B <= 16 && deep && V >= 65536;
  const bool staged1 = wide1 && B >= 10 && K % 2048 != 0 && fills(32768);
  const bool tall = wide1 && !staged1 && B >= 11 && fills(16384);
  const int nt = staged1 ? 2 : (B + 15) / 16;
  const bool split = nt == 1 || V <= (nt == 2 ? 14336 : 9216);
  const int rows = split ? (tall ? 64 : 32) : HG_W * HG_MT * 16;
  const dim3 grid((unsigned)((V + rows - 1) / rows));
#define STRIM_HEAD_(K_, NT_, MT_, NW_, VO_, TB_)                                              \
  hipLaunchKernelGGL((K_<NT_, VO_, TB_, MT_, NW_>), grid, dim3(NW_ * WAVE), 0, st, src,       \
                     src_stride, B, K, (const uint16_t*)W, w_stride, V, (uint16_t*)out,       \
                     out_stride, tbest)
#define STRIM_HEAD(K_, NT_, MT_, NW_)                             \
  do {                                                            \
    if (tbest && vo) STRIM_HEAD_(K_, NT_, MT_, NW_, true, true);  \
    else if (tbest) STRIM_HEAD_(K_, NT_, MT_, NW_, false, true);  \
    else if (vo) STRIM_HEAD_(K_, NT_, MT_, NW_, true, false);     \
    else STRIM_HEAD_(K_, NT_, MT_, NW_, false, false);            \
  } while (0)
  if (tall) STRIM_HEAD(k_head_split, 1, 4, 8);
  else if (nt == 1 && deep) STRIM_HEAD(k_head_split, 1, 2, 8);
  else if (nt == 1) STRIM_HEAD(k_head_split, 1, 2, 4);
  else if (nt == 2 && split && deep) STRIM_HEAD(k_head_split, 2, 2, 8);
  else if (nt == 2 && split) STRIM_HEAD(k_head_split, 2, 2, 4);
  else if (nt == 2) STRIM_HEAD(k_head_gemv, 2, HG_MT, HG_W);
  else if (split && deep) STRIM_HEAD(k_head_split, 4, 2, 8);
  else if (split) STRIM_HEAD(k_head_split, 4, 2, 4);
  else STRIM_HEAD(k_head_gemv, 4, HG_MT, HG_W);
#undef STRIM_HEAD
#undef STRIM_HEAD_
  if (tbest)
    hipLaunchKernelGGL(k_head_pick, dim3((unsigned)B), dim3(HP_T), 0, st, tbest, (int)grid.x,
                       out_ids, out_status);
  return hipGetLastError();
}

}  // namespace strim
