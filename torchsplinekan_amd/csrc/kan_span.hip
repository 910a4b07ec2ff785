// Span-window products: the fp32 forward product and the input gradient of a
// layer with many basis functions per feature, on the k + 1 that are not zero.
//
// A dense product over H's columns costs R + 1 multiply-adds per (sample,
// feature, output); a sample's row holds k + 1 values per feature and its
// SiLU, so k + 2 suffice.  These kernels take x instead of H: a lane evaluates
// one (sample, feature) item, and its wave then walks the items, each one
// reading the k + 1 weight rows of its span from LDS, which is the transposed
// augmented weight Wt [I R + I, O] (rows of O, feature-major):
//   forward   y[n, o]  = sum_i ( sum_j B_j(x) Wt[i R + m - k + j, o] + silu(x) Wt[I R + i, o] )
//   input     dx[n, i] = sum_o D[n, o] ( sum_j B'_j(x) Wt[i R + m - k + j, o]
//                                        + silu'(x) Wt[I R + i, o] )
// (m the span of x[n, i]; nothing from the spline where x is outside its knots)
// with fp32 FMAs in a fixed order: the features of a slice one after the
// other, the slices' sums in order.
//
// What bounds it: LDS reads and VALU issue together.  An item and 256 outputs
// take 4 KB of LDS reads (32 clocks of a CU at k = 3) and 27 VALU operations a
// wave (27 clocks; 37 for the input gradient), and two waves per SIMD overlap
// the two by half: 64 and 74 clocks measured.  At 8192 x 4096 -> 256, R = 68:
// forward 3.65 ms against 5.10 ms for the split-bf16 product over all columns
// (which also needs the basis written, 1.73 ms), input gradient 4.23 against
// 7.31 + 0.33 ms (compact product and its window pass), timed alone (3.9 and
// 4.4 ms within a training step).
//
// Layout: 8 waves of 24 (input: 20) samples share the weight rows of one feature and
// 64 V outputs (V per lane), double buffered in LDS while the next feature's
// are in flight in registers; K zero rows on either side of the feature's R
// stand for window entries that are no basis function.  The accumulators
// (forward) or dL/dy (input) of the wave's block stay in registers.

#include <type_traits>

#include "kan_common.h"
#include "kan_spline.h"

namespace kan {
namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kSpanWaves = 8;
constexpr int kSpanThreads = 64 * kSpanWaves;
// Samples per wave: as many as leave the registers of a 256-output block
// unspilled (at most 32, a half's lanes).  With 32 the staged rows spill, and
// a reload waits for the loads in flight: 4.29 against 3.65 ms forward, 4.81
// against 4.23 ms for the input gradient at 8192 x 4096 -> 256, R = 68.
constexpr int span_samples(bool dx) { return dx ? 20 : 24; }
// Samples per block.
constexpr int span_tile(bool dx) { return kSpanWaves * span_samples(dx); }
constexpr int kSpanChunk = 8;                     // features: granule of a slice
constexpr int kSpanGroup = 1;                     // samples whose LDS reads are in flight together

struct SpanParams {
  const float* x;
  const float* grid;
  const float* wt;   // [I R (+ I), O]
  const float* D;    // input gradient: dL/dy [n, O]
  float* out;        // forward: [slices][n, O]; input: [output tiles][n, I]
  int64_t n, I, O;
  int64_t feats;     // features per slice (a multiple of kSpanChunk)
  int64_t out_stride;
  int R, nk, base;
  int tiles_n, tiles_o, slices;
};

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

template <int V>
struct SpanVec {
  typedef float type __attribute__((ext_vector_type(V)));
};
template <>
struct SpanVec<1> {
  typedef float type;
};
template <int V>
__device__ __forceinline__ float vec_at(const typename SpanVec<V>::type& v, int j) {
  if constexpr (V == 1) return v;
  else return v[j];
}

template <int K, int V, bool DX>
__global__ __launch_bounds__(kSpanThreads) __attribute__((amdgpu_waves_per_eu(V == 4 ? 2 : V == 2 ? 3 : 4))) void
span_kernel(SpanParams p) {
  typedef typename SpanVec<V>::type vec_t;
  constexpr int kSpanS = span_samples(DX);
  constexpr int OB = 64 * V;                       // outputs per block
  constexpr int kGroups = OB / 4;                  // 16-byte column groups
  constexpr int kRowsPer = kSpanThreads / kGroups; // slab rows a pass of the block covers
  constexpr int kLoads = (kMaxR + kRowsPer - 1) / kRowsPer;
  extern __shared__ __align__(16) float lds[];
  const int R = p.R, nk = p.nk;
  const int slab = (R + 2 * K + 1) * OB;           // pads, R rows, pads, base row
  float* const wbuf0 = lds;
  float* const kbuf0 = lds + 2 * slab;             // [2][2][nk]

  const int total = p.tiles_n * p.tiles_o * p.slices;
  const int pid = xcd_remap(blockIdx.x, total);    // blocks of one slice share an L2
  const int tn = __builtin_amdgcn_readfirstlane(pid % p.tiles_n);
  const int rest = __builtin_amdgcn_readfirstlane(pid / p.tiles_n);
  const int slice = __builtin_amdgcn_readfirstlane(rest % p.slices);
  const int to = __builtin_amdgcn_readfirstlane(rest / p.slices);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int64_t o0 = (int64_t)to * OB;
  const int64_t n0 = (int64_t)tn * span_tile(DX) + wave * kSpanS;
  const int64_t fbeg = (int64_t)slice * p.feats, fend = min(p.I, fbeg + p.feats);
  const int half = lane >> 5;
  const int64_t ns = min(n0 + min(lane & 31, kSpanS - 1), p.n - 1);  // this lane's sample

  // staging of one feature's rows: thread -> column group g, rows r0, r0 + kRowsPer, ...
  const int cg = threadIdx.x % kGroups, r0 = threadIdx.x / kGroups;
  const int64_t oc = o0 + 4 * cg;
  const bool vec = (p.O & 3) == 0;
  u32x4 st[kLoads], sb;  // the R rows, and (threads of row 0) the base row
  float poison[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  // Branch-free buffer loads: an offset past the resource reads as zero (rows
  // past R, columns past O).  A load under a condition makes the compiler
  // wait for it where the branches join, one row after the other: 5.91
  // against 4.81 ms for the input gradient at 8192 x 4096 -> 256, R = 68.
  const uint32_t step = (uint32_t)(kRowsPer * p.O * 4);
  const auto rsrc = [&](const float* base) __attribute__((always_inline)) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), (short)0, 0x7fffffff,
                                             0x00020000 /* raw buffer, 32-bit data */);
  };
  auto load_rows = [&](int64_t f) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rs = rsrc(p.wt + f * R * p.O + o0);
    const __amdgpu_buffer_rsrc_t rb = rsrc(p.wt + (p.I * R + f) * p.O + o0);
    const uint32_t at = (uint32_t)(((int64_t)r0 * p.O + 4 * cg) * 4);
    if (vec) {
#pragma unroll
      for (int u = 0; u < kLoads; ++u) {
        const bool in = r0 + u * kRowsPer < R && oc < p.O;
        st[u] = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(in ? at + u * step : 0x80000000u), 0, 0);
      }
      const bool in = p.base && r0 == 0 && oc < p.O;
      sb = __builtin_amdgcn_raw_buffer_load_b128(rb, (int)(in ? (uint32_t)(16 * cg) : 0x80000000u), 0, 0);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
          const bool in = r0 + u * kRowsPer < R && oc + j < p.O;
          st[u][j] = __builtin_amdgcn_raw_buffer_load_b32(
              rs, (int)(in ? at + u * step + 4 * j : 0x80000000u), 0, 0);
        }
        const bool in = p.base && r0 == 0 && oc + j < p.O;
        sb[j] = __builtin_amdgcn_raw_buffer_load_b32(
            rb, (int)(in ? (uint32_t)(16 * cg + 4 * j) : 0x80000000u), 0, 0);
      }
    }
  };
  auto store_rows = [&](float* buf) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int r = r0 + u * kRowsPer;
      if (r < R) *reinterpret_cast<u32x4*>(buf + (K + r) * OB + 4 * cg) = st[u];
    }
    if (r0 == 0) *reinterpret_cast<u32x4*>(buf + (R + 2 * K) * OB + 4 * cg) = sb;
    if constexpr (!DX) {
      // (NaN where a spline weight is not finite: see the end)
#pragma unroll
      for (int u = 0; u < kLoads; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          poison[j] = __builtin_fmaf(__uint_as_float(st[u][j]), 0.0f, poison[j]);
    }
  };

  // forward: sums of the block's samples; input: dL/dy of them
  float blk[kSpanS][V];
#pragma unroll
  for (int s = 0; s < kSpanS; ++s) {
    const int64_t n = min(n0 + s, p.n - 1);
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int64_t o = o0 + lane * V + v;
      blk[s][v] = DX && o < p.O ? p.D[n * p.O + o] : 0.0f;
    }
  }

  // zero rows of both buffers (never written again), then the first feature
  for (int e = threadIdx.x; e < 2 * 2 * K * OB; e += kSpanThreads) {
    const int b = e / (2 * K * OB), q = e - b * (2 * K * OB);
    const int r = q / OB, c = q - r * OB;
    wbuf0[b * slab + (r < K ? r : R + r) * OB + c] = 0.0f;
  }
  float xv = 0.0f;
  if (fbeg < fend) {
    load_rows(fbeg);
    store_rows(wbuf0);
    for (int e = threadIdx.x; e < 2 * nk; e += kSpanThreads)
      if (fbeg * nk + e < fend * nk) kbuf0[e] = p.grid[fbeg * nk + e];
    xv = p.x[ns * p.I + min(fbeg + half, fend - 1)];
  }
  int t = 0;  // features done: buffer t & 1
#pragma unroll 1
  for (int64_t f0 = fbeg; f0 < fend; f0 += 2) {
    // two features: lanes 0-31 evaluate the first, lanes 32-63 the second;
    // the next pair's knots and x are on their way meanwhile
    const int par = (int)((f0 - fbeg) >> 1) & 1;
    const float* kn = kbuf0 + par * 2 * nk;
    const float kreg = p.grid[min((f0 + 2) * nk + threadIdx.x, fend * nk - 1)];
    const float xnext = p.x[ns * p.I + min(f0 + 2 + half, fend - 1)];
    float b[K + 1], sl = 0.0f;
    int mrow = 0;
    float res = 0.0f;
#pragma unroll 1
    for (int h = 0; h < 2 && f0 + h < fend; ++h) {
      __syncthreads();  // this feature's rows (and knots) are in LDS; the other buffer is free
      const bool more = f0 + h + 1 < fend;
      if (more) load_rows(f0 + h + 1);
      if (h == 0) {
        const float* tk = kn + (f0 + half < fend ? half : 0) * nk;
        int m = knot_span(tk, nk, xv);
        const bool in = m >= 0;
        if (!in) m = K;
        if constexpr (DX) span_derivs<K, float>(tk, nk, m, xv, b);
        else span_values<K, float>(tk, nk, m, xv, b);
#pragma unroll
        for (int j = 0; j <= K; ++j) {
          const int r = m - K + j;
          if (!in || r < 0 || r >= R) b[j] = 0.0f;
        }
        mrow = m * OB;  // window entry j lies in slab row m + j
        if (p.base) sl = DX ? silu_grad_of<float>(xv) : silu_of<float>(xv);
      }
      const float* buf = wbuf0 + (t & 1) * slab + lane * V;
      const vec_t wb = *reinterpret_cast<const vec_t*>(buf + (R + 2 * K) * OB);
      int h32 = h * 32;
      float part[DX ? 32 : 1];
      if constexpr (DX) {
#pragma unroll
        for (int s = kSpanS; s < 32; ++s) part[s] = 0.0f;
      }
      // kSpanGroup samples at a time, the next group's rows on their way from
      // LDS while this one's arithmetic runs
      float cs[2][kSpanGroup][K + 1], sv[2][kSpanGroup];
      vec_t w[2][kSpanGroup][K + 1];
      auto fetch = [&](int g, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < kSpanGroup; ++u) {
          const int src = h32 + g * kSpanGroup + u;
          const float* wr = buf + __builtin_amdgcn_readlane(mrow, src);
#pragma unroll
          for (int j = 0; j <= K; ++j) w[slot][u][j] = *reinterpret_cast<const vec_t*>(wr + j * OB);
          sv[slot][u] = lane_value(sl, src);
#pragma unroll
          for (int j = 0; j <= K; ++j) cs[slot][u][j] = lane_value(b[j], src);
        }
      };
      fetch(0, 0);
#pragma unroll
      for (int g = 0; g < kSpanS / kSpanGroup; ++g) {
        // (without the fences the lane reads and loads of every sample come
        // first, and spill)
        asm volatile("" : "+s"(h32) : : "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (g + 1 < kSpanS / kSpanGroup) fetch(g + 1, (g + 1) & 1);
#pragma unroll
        for (int u = 0; u < kSpanGroup; ++u) {
          const int s = g * kSpanGroup + u, slot = g & 1;
          if constexpr (DX) {
            float dot = 0.0f;
#pragma unroll
            for (int v = 0; v < V; ++v) {
              float q = sv[slot][u] * vec_at<V>(wb, v);
#pragma unroll
              for (int j = 0; j <= K; ++j)
                q = __builtin_fmaf(cs[slot][u][j], vec_at<V>(w[slot][u][j], v), q);
              dot = __builtin_fmaf(blk[s][v], q, dot);
            }
            asm volatile("" : "+v"(dot));
            part[s] = dot;
          } else {
#pragma unroll
            for (int v = 0; v < V; ++v) {
              float q = __builtin_fmaf(sv[slot][u], vec_at<V>(wb, v), blk[s][v]);
#pragma unroll
              for (int j = 0; j <= K; ++j)
                q = __builtin_fmaf(cs[slot][u][j], vec_at<V>(w[slot][u][j], v), q);
              // (pinned here: the sum's next use is in the next iteration, and
              // the compiler would sink its arithmetic past the branches below,
              // keeping every sample's operands in registers)
              asm volatile("" : "+v"(q));
              blk[s][v] = q;
            }
          }
        }
      }
      if constexpr (DX) {
        // sums over the 64 lanes: after the five exchanges lane l holds
        // sample l & 31's sum over 32 lanes, then the other half's is added
#pragma unroll
        for (int lv = 0; lv < 5; ++lv) {
          const bool up = (lane >> lv) & 1;
#pragma unroll
          for (int q = 0; q < (32 >> (lv + 1)); ++q) {
            const float a = part[2 * q], c = part[2 * q + 1];
            part[q] = (up ? c : a) + __shfl_xor(up ? a : c, 1 << lv);
          }
        }
        const float sum = part[0] + __shfl_xor(part[0], 32);
        if (half == h) res = sum;
      }
      // (the next feature's rows go to the buffer that no wave reads now)
      if (more) store_rows(wbuf0 + ((t + 1) & 1) * slab);
      ++t;
    }
    if ((int)threadIdx.x < 2 * nk) kbuf0[(par ^ 1) * 2 * nk + threadIdx.x] = kreg;
    xv = xnext;
    if constexpr (DX) {
      if ((lane & 31) < kSpanS && n0 + (lane & 31) < p.n && f0 + half < fend)
        p.out[(int64_t)to * p.out_stride + (n0 + (lane & 31)) * p.I + f0 + half] = res;
    }
  }
  if constexpr (!DX) {
    // A spline weight that is not finite meets every sample in the dense
    // product: times a basis value where the sample's window holds it (the
    // loop above), times 0 elsewhere.  A block that staged one adds these
    // zeros' products here, so that infinities and NaN come out as they do
    // there.  (The base weights met every sample above.)
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) lds[r0 * OB + 4 * cg + j] = poison[j];
    __syncthreads();
    float any = 0.0f;
#pragma unroll
    for (int v = 0; v < V; ++v)
      for (int r = 0; r < kRowsPer; ++r) any += lds[r * OB + lane * V + v];
    if (__any(any != 0.0f)) {
#pragma unroll 1
      for (int64_t f = fbeg; f < fend; ++f) {
        const int m = knot_span(p.grid + f * nk, nk, p.x[ns * p.I + f]);
#pragma unroll 1
        for (int r = 0; r < R; ++r) {
          float z[V];  // 0, or NaN
          bool bad = false;
#pragma unroll
          for (int v = 0; v < V; ++v) {
            const int64_t o = o0 + lane * V + v;
            z[v] = o < p.O ? p.wt[(f * R + r) * p.O + o] * 0.0f : 0.0f;
            bad |= z[v] != 0.0f;
          }
          if (!__any(bad)) continue;
#pragma unroll
          for (int s = 0; s < kSpanS; ++s) {
            const int ms = __builtin_amdgcn_readlane(m, s);
            if (ms >= 0 && r >= ms - K && r <= ms) continue;
#pragma unroll
            for (int v = 0; v < V; ++v) blk[s][v] += z[v];
          }
        }
      }
    }
    float* out = p.out + (int64_t)slice * p.out_stride;
#pragma unroll
    for (int s = 0; s < kSpanS; ++s) {
      if (n0 + s >= p.n) continue;
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const int64_t o = o0 + lane * V + v;
        if (o < p.O) out[(n0 + s) * p.O + o] = blk[s][v];
      }
    }
  }
}

// wt[c, o] = w[o, c] for c < kaug (the packed inference weight's rows of ld)
constexpr int kTr = 64;
__global__ __launch_bounds__(256) void transpose_kernel(const float* __restrict__ w, int64_t ld,
                                                       float* __restrict__ wt, int64_t O,
                                                       int64_t kaug) {
  __shared__ float tile[kTr][kTr + 1];
  const int64_t c0 = (int64_t)blockIdx.x * kTr, o0 = (int64_t)blockIdx.y * kTr;
  const int l = threadIdx.x & 63, w4 = threadIdx.x >> 6;
  for (int r = w4; r < kTr; r += 4)
    if (o0 + r < O && c0 + l < kaug) tile[r][l] = w[(o0 + r) * ld + c0 + l];
  __syncthreads();
  for (int r = w4; r < kTr; r += 4)
    if (c0 + r < kaug && o0 + l < O) wt[(c0 + r) * O + o0 + l] = tile[l][r];
}

// out[e] = sum_s part[s][e], s in order
__global__ void span_sum_kernel(const float* __restrict__ part, int slices, int64_t count,
                                float* __restrict__ out) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < count;
       e += (int64_t)gridDim.x * blockDim.x) {
    float v = part[e];
    for (int s = 1; s < slices; s += 4) {
      float w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = part[min(s + u, slices - 1) * count + e];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (s + u < slices) v += w[u];
    }
    out[e] = v;
  }
}

// The input gradient's items that came out infinite or NaN, evaluated again in
// the dense product's order: each weight row of the item's window summed over
// the outputs, then times its derivative.  The span kernel's sums differ there
// (0 times such a value, the rows it reads for an x outside the knots,
// infinities of both signs).  A wave looks through 256 items at a time and
// takes a bad one with all its lanes; where there is none the pass costs its
// reads (a kernel of its own, since the span kernel has no register left: the
// same check at its end took 3 % of it, the pass takes 1 %).
constexpr int kAgainItems = 4;  // per lane
template <int K>
__global__ __launch_bounds__(256) void span_dx_again_kernel(SpanParams p, float* __restrict__ gx) {
  const int lane = threadIdx.x & 63;
  const int64_t count = p.n * p.I, step = (int64_t)gridDim.x * 256 * kAgainItems;
  const int64_t first = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 64 * kAgainItems;
#pragma unroll 1
  for (int64_t e0 = first; e0 < count; e0 += step) {
    float v[kAgainItems];
#pragma unroll
    for (int u = 0; u < kAgainItems; ++u) {
      const int64_t e = e0 + 64 * u + lane;
      v[u] = e < count ? gx[e] : 0.0f;
    }
#pragma unroll 1
    for (int u = 0; u < kAgainItems; ++u) {
      uint64_t again = __ballot(v[0] * 0.0f != 0.0f);
#pragma unroll
      for (int w = 0; w + 1 < kAgainItems; ++w) v[w] = v[w + 1];
#pragma unroll 1
      for (; again != 0; again &= again - 1) {
        const int64_t e = e0 + 64 * u + __builtin_ctzll(again);
        const int64_t n = e / p.I, f = e - n * p.I;
        const float* tk = p.grid + f * p.nk;
        const float xv = p.x[e];
        const int m = knot_span(tk, p.nk, xv);
        float b[K + 1];
        span_derivs<K, float>(tk, p.nk, m >= 0 ? m : K, xv, b);
        auto row_sum = [&](int64_t row) {
          float a = 0.0f;
          for (int64_t o = lane; o < p.O; o += 64)
            a = __builtin_fmaf(p.D[n * p.O + o], p.wt[row * p.O + o], a);
#pragma unroll
          for (int off = 32; off >= 1; off >>= 1) a += __shfl_xor(a, off);
          return a;
        };
        float q = 0.0f;
#pragma unroll
        for (int j = 0; j <= K; ++j) {
          const int r = m - K + j;
          if (m >= 0 && r >= 0 && r < p.R) q += row_sum(f * p.R + r) * b[j];
        }
        if (p.base) q += row_sum(p.I * p.R + f) * silu_grad_of<float>(xv);
        if (lane == 0) gx[e] = q;
      }
    }
  }
}

size_t span_lds_bytes(int K, int V, int R, int nk) {
  const size_t need = sizeof(float) * (2 * (size_t)(R + 2 * K + 1) * 64 * V + 4 * (size_t)nk);
  return std::max(need, sizeof(float) * 4 * (size_t)kSpanThreads);  // (the poison's reduction)
}

template <int K, int V, bool DX>
int launch_span_kv(const SpanParams& p, hipStream_t st) {
  const size_t bytes = span_lds_bytes(K, V, p.R, p.nk);
  static_assert(sizeof(float) * (2 * (kMaxR + 2 * 3 + 1) * 256 + 4 * kMaxKnots) <=
                    160 * 1024,
                "the widest rows fit the LDS");
  const hipError_t e = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&span_kernel<K, V, DX>),
      hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (e != hipSuccess)
    return set_error(KAN_ERR_HIP, "span product: %zu bytes of LDS: %s", bytes, hipGetErrorString(e));
  const int64_t blocks = (int64_t)p.tiles_n * p.tiles_o * p.slices;
  hipLaunchKernelGGL((span_kernel<K, V, DX>), dim3((unsigned)blocks), dim3(kSpanThreads), bytes,
                     st, p);
  return check_launch("span product");
}

template <bool DX>
int launch_span(const SpanParams& p, int k, int V, hipStream_t st) {
#define KAN_SPAN(KK)                                             \
  do {                                                           \
    if (V == 4) return launch_span_kv<KK, 4, DX>(p, st);         \
    if (V == 2) return launch_span_kv<KK, 2, DX>(p, st);         \
    return launch_span_kv<KK, 1, DX>(p, st);                     \
  } while (0)
  if (k == 1) KAN_SPAN(1);
  if (k == 2) KAN_SPAN(2);
  KAN_SPAN(3);
#undef KAN_SPAN
}

// Clocks (at 2.3 GHz) a CU takes per (sample, feature) item and output tile of
// 64 V, measured at k = 3 from 16 to 68 basis functions (within 8 %).
double span_clocks(int V, bool dx) {
  return V == 4 ? (dx ? 74.0 : 64.0) : V == 2 ? (dx ? 55.0 : 44.0) : (dx ? 36.0 : 28.0);
}

}  // namespace

// Outputs per lane and feature slices: the outputs' tiles with the fewest
// clocks, then the slice count whose blocks fill whole rounds of the CUs best
// (one block per CU; a slice's start-up and, forward, its sum's traffic as
// 2 % of a round each).
SpanPlan span_plan(int64_t n, int64_t I, int64_t O, int64_t R, int64_t k, bool dx) {
  SpanPlan p{};
  const int64_t cus = device_cu_count();
  const int64_t tn = ceil_div(n, (int64_t)span_tile(dx));
  double best_v = 0.0;
  for (int V : {4, 2, 1}) {
    const double c = (double)ceil_div(O, (int64_t)(64 * V)) * span_clocks(V, dx);
    if (p.v == 0 || c < best_v) {
      p.v = V;
      best_v = c;
    }
  }
  p.tiles_n = tn;
  p.tiles_o = ceil_div(O, (int64_t)(64 * p.v));
  const int64_t chunks = ceil_div(I, (int64_t)kSpanChunk);
  double best = 0.0;
  // (forward slices leave partial sums: at most 24 of them, and no more than
  // the basis would take)
  for (int64_t s = 1; s <= (dx ? 64 : 24) && s <= chunks; ++s) {
    if (!dx && s > 1 && s * O > I * (R + 1)) break;
    const int64_t per = ceil_div(chunks, s);
    if (s > 1 && (per < 4 || ceil_div(chunks, per) != s)) continue;
    const double rounds = (double)ceil_div(p.tiles_n * p.tiles_o * s, cus);
    const double items = rounds * (double)per * kSpanChunk * span_tile(dx) * span_clocks(p.v, dx);
    // clocks at 2.3 GHz; slices' partial sums (forward) at 5 TB/s
    const double sum = !dx && s > 1 ? 8.0 * (double)s * (double)(n * O) / 5e12 : 0.0;
    const double t = items / 2.3e9 + rounds * 6e-6 + sum;
    if (p.slices == 0 || t < best) {
      best = t;
      p.slices = s;
      p.feats = per * kSpanChunk;
    }
  }
  if (p.slices == 0) {
    p.slices = 1;
    p.feats = chunks * kSpanChunk;
  }
  p.seconds = best;
  const int64_t parts = dx ? p.tiles_o : p.slices;
  p.part_elems = parts > 1 ? parts * n * (dx ? I : O) : 0;
  if (dx && parts > 1) p.seconds += 8.0 * (double)p.part_elems / 5e12;
  (void)k;
  return p;
}

namespace {
SpanParams span_params(const SpanPlan& pl, const float* x, const float* grid, const float* wt,
                       int64_t n, int64_t I, int64_t O, int G, int k, bool base) {
  SpanParams p{};
  p.x = x;
  p.grid = grid;
  p.wt = wt;
  p.n = n;
  p.I = I;
  p.O = O;
  p.feats = pl.feats;
  p.R = G + k;
  p.nk = G + 2 * k + 1;
  p.base = base ? 1 : 0;
  p.tiles_n = (int)pl.tiles_n;
  p.tiles_o = (int)pl.tiles_o;
  p.slices = (int)pl.slices;
  return p;
}

int sum_parts(const float* part, int64_t parts, int64_t count, float* out, hipStream_t st) {
  const unsigned blocks = (unsigned)std::min<int64_t>(ceil_div(count, (int64_t)256), 65536);
  hipLaunchKernelGGL(span_sum_kernel, dim3(blocks), dim3(256), 0, st, part, (int)parts, count, out);
  return check_launch("span sum");
}
}  // namespace

int launch_span_forward(const SpanPlan& pl, const float* x, const float* grid, const float* wt,
                        float* y, float* part, int64_t n, int64_t I, int64_t O, int G, int k,
                        bool base, hipStream_t st) {
  SpanParams p = span_params(pl, x, grid, wt, n, I, O, G, k, base);
  p.out = pl.slices > 1 ? part : y;
  p.out_stride = n * O;
  {
    TimedLaunch timed(kClassContraction, st,
                      2.0 * (double)n * (double)O * (double)I * (k + 1 + (base ? 1 : 0)));
    const int rc = launch_span<false>(p, k, pl.v, st);
    if (rc != KAN_OK) return rc;
  }
  return pl.slices > 1 ? sum_parts(part, pl.slices, n * O, y, st) : KAN_OK;
}

int launch_span_dx(const SpanPlan& pl, const float* D, const float* x, const float* grid,
                   const float* wt, float* gx, float* part, int64_t n, int64_t I, int64_t O, int G,
                   int k, bool base, hipStream_t st) {
  SpanParams p = span_params(pl, x, grid, wt, n, I, O, G, k, base);
  p.D = D;
  p.out = pl.tiles_o > 1 ? part : gx;
  p.out_stride = n * I;
  {
    TimedLaunch timed(kClassContraction, st,
                      2.0 * (double)n * (double)O * (double)I * (k + 1 + (base ? 1 : 0)));
    const int rc = launch_span<true>(p, k, pl.v, st);
    if (rc != KAN_OK) return rc;
  }
  if (pl.tiles_o > 1) {
    const int rc = sum_parts(part, pl.tiles_o, n * I, gx, st);
    if (rc != KAN_OK) return rc;
  }
  TimedLaunch timed(kClassOther, st, 0.0);
  const dim3 blocks((unsigned)std::min<int64_t>(ceil_div(n * I, (int64_t)(256 * kAgainItems)), 4096));
  if (k == 1) hipLaunchKernelGGL(span_dx_again_kernel<1>, blocks, dim3(256), 0, st, p, gx);
  else if (k == 2) hipLaunchKernelGGL(span_dx_again_kernel<2>, blocks, dim3(256), 0, st, p, gx);
  else hipLaunchKernelGGL(span_dx_again_kernel<3>, blocks, dim3(256), 0, st, p, gx);
  return check_launch("span input gradient, values that are not finite");
}

int launch_transpose(const float* w, int64_t ld, float* wt, int64_t O, int64_t kaug,
                     hipStream_t st) {
  TimedLaunch timed(kClassOther, st, 0.0);
  hipLaunchKernelGGL(transpose_kernel,
                     dim3((unsigned)ceil_div(kaug, (int64_t)kTr), (unsigned)ceil_div(O, (int64_t)kTr)),
                     dim3(256), 0, st, w, ld, wt, O, kaug);
  return check_launch("transpose");
}

}  // namespace kan
