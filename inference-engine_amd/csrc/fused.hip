// fused.hip — gfx950 element-wise kernels beside the paged-KV path: the RMSNorm tail,
// in-place RoPE and SiLU-and-multiply, each one launch instead of PyTorch's chain of
// small kernels, 16 bytes per access where pointers, strides and widths allow (one
// element per thread otherwise). C ABI in include/paged_kv.h.
//
// Each kernel rounds exactly where the PyTorch ops it replaces round, so results are
// bitwise identical to them: every product and sum is one fp32 operation rounded to the
// tensor dtype at the points PyTorch rounds, exp and division are the device library's
// and IEEE (as in PyTorch's ROCm SiLU), and multiply-add contraction is off for the whole
// file (PyTorch's separate kernels round between the multiply and the add). RMSNorm leaves
// the mean of its squares to PyTorch (a sum in another order has other bits); its rsqrt is
// 1 / sqrt(x) in fp64 rounded to fp32, which is what PyTorch's ROCm rsqrt gives on every
// non-negative fp32 value (the device library's rsqrtf differs on 11% of them).

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "paged_kv.h"

#pragma clang fp contract(off)

namespace {

template <int DT> struct F;
template <> struct F<PKV_F32> {
  using S = float;
  __device__ static float up(S x) { return x; }
  __device__ static S down(float f) { return f; }
};
template <> struct F<PKV_F16> {
  using S = uint16_t;
  __device__ static float up(S x) { return (float)__builtin_bit_cast(_Float16, x); }
  // v_cvt_f16_f32, round to nearest even; the empty asm keeps f an fp32 value (no fused
  // multiply-and-convert, which would round once instead of twice).
  __device__ static S down(float f) {
    __asm__ volatile("" : "+v"(f));
    return __builtin_bit_cast(uint16_t, (_Float16)f);
  }
};
template <> struct F<PKV_BF16> {
  using S = uint16_t;
  __device__ static float up(S x) { return __uint_as_float(uint32_t(x) << 16); }
  // Round to nearest even on the upper half; NaN becomes 0x7FC0 (torch's float ->
  // bfloat16).
  __device__ static S down(float f) {
    if (f != f) return 0x7FC0;
    const uint32_t u = __float_as_uint(f);
    return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
  }
};

// Value as it is after a cast to DT and back to fp32.
template <int DT> __device__ __forceinline__ float through(float f) {
  return F<DT>::up(F<DT>::down(f));
}

// 16 bytes of DT: VN<DT> elements (8 of a 16-bit type, 4 floats).
template <int DT> constexpr int VN = DT == PKV_F32 ? 4 : 8;
// NT: non-temporal, for data too large to be found in the caches again.
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
template <int DT, bool NT = false>
__device__ __forceinline__ void load16(const typename F<DT>::S* p, float* f) {
  const u32x4* q = reinterpret_cast<const u32x4*>(p);
  const u32x4 r = NT ? __builtin_nontemporal_load(q) : *q;
  const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (DT == PKV_F32) {
      f[i] = __uint_as_float(w[i]);
    } else {
      f[2 * i] = F<DT>::up((uint16_t)(w[i] & 0xFFFFu));
      f[2 * i + 1] = F<DT>::up((uint16_t)(w[i] >> 16));
    }
  }
}
// Two values rounded to a 16-bit DT, packed. bf16 through v_cvt_pk_bf16_f32, which rounds every
// value as down() does but keeps the bits of a NaN.
template <int DT> __device__ __forceinline__ uint32_t pack2(float a, float b) {
  if constexpr (DT == PKV_BF16) {
    typedef __bf16 v2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, v2{(__bf16)a, (__bf16)b});
  } else {
    return (uint32_t)F<DT>::down(a) | ((uint32_t)F<DT>::down(b) << 16);
  }
}
// f[0 .. N) after a cast to DT and back (through()), in place; the bits of NaNs aside, which
// the store of whatever is computed from them sets.
template <int DT, int N> __device__ __forceinline__ void round_all(float* f) {
  if constexpr (DT != PKV_F32) {
#pragma unroll
    for (int i = 0; i < N; i += 2) {
      const uint32_t w = pack2<DT>(f[i], f[i + 1]);
      f[i] = F<DT>::up((uint16_t)(w & 0xFFFFu));
      f[i + 1] = F<DT>::up((uint16_t)(w >> 16));
    }
  }
}
template <int DT, bool NT = false>
__device__ __forceinline__ void store16(typename F<DT>::S* p, const float* f) {
  uint32_t w[4];
  if constexpr (DT == PKV_F32) {
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = __float_as_uint(f[i]);
  } else {
    bool nan = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      w[i] = pack2<DT>(f[2 * i], f[2 * i + 1]);
      nan = nan || __builtin_isunordered(f[2 * i], f[2 * i + 1]);
    }
    if (DT == PKV_BF16 && nan) {  // PyTorch's one NaN
#pragma unroll
      for (int i = 0; i < 4; ++i)
        w[i] = (uint32_t)F<DT>::down(f[2 * i]) | ((uint32_t)F<DT>::down(f[2 * i + 1]) << 16);
    }
  }
  u32x4* q = reinterpret_cast<u32x4*>(p);
  const u32x4 v = {w[0], w[1], w[2], w[3]};
  if constexpr (NT) __builtin_nontemporal_store(v, q);
  else *q = v;
}
// n fp32 values (n a multiple of 4) from a 16-byte aligned address.
template <int N> __device__ __forceinline__ void load_f32(const float* p, float* f) {
#pragma unroll
  for (int i = 0; i < N; i += 4) {
    const float4 v = *reinterpret_cast<const float4*>(p + i);
    f[i] = v.x, f[i + 1] = v.y, f[i + 2] = v.z, f[i + 3] = v.w;
  }
}

// A row's scale: the caller's inv_rms, or rsqrt(mean + eps) from its mean of squares.
struct RowScale {
  const float* v;
  float eps;
  bool mean;
  __device__ __forceinline__ float at(int64_t r) const {
    return mean ? (float)(1.0 / sqrt((double)(v[r] + eps))) : v[r];
  }
};

// Rows of n elements (or vectors) on workgroups of 256: 2^lg threads side by side take a row, so
// a workgroup takes 256 >> lg rows at once. With a workgroup per row, rows of 8 to 128 elements
// kept 1 to 32 of its threads (RMSNorm of 300,000 rows of 8, bf16: 212.7 us, now 22.0; 69,376 of
// 128: 84.8, now 30.8).
// WHOLE: a row takes the whole workgroup, known at compile time, so its number and mean are
// scalars (2,168 rows of 4,099, one element per access: 50.1 us against 53.4).
template <bool WHOLE> struct RowLanes {
  int lg_;
  explicit RowLanes(int n) : lg_(0) {
    while (lg_ < 8 && (1 << lg_) < n) ++lg_;
  }
  __host__ __device__ __forceinline__ int lg() const { return WHOLE ? 8 : lg_; }
  __host__ __device__ __forceinline__ int per_wg() const { return 256 >> lg(); }
  __device__ __forceinline__ int sub() const { return WHOLE ? 0 : (int)threadIdx.x >> lg_; }  // which row
  __device__ __forceinline__ int lane() const {
    return WHOLE ? (int)threadIdx.x : (int)threadIdx.x & ((1 << lg_) - 1);
  }
};

// out[r, c] = DO( f32(w[c]) * f32(DX( f32(x[r, c]) * inv[r] )) ): PyTorch's
// w * (x.float() * inv).to(x.dtype), inv = torch.rsqrt(mean(x.float()^2) + eps) per row.
template <int DX, int DW, int DO, bool WHOLE>
__global__ void __launch_bounds__(256)
rms_norm_tail_kernel(typename F<DO>::S* __restrict__ out, int64_t so,
                     const typename F<DX>::S* __restrict__ x, int64_t sx, const RowScale scale,
                     const typename F<DW>::S* __restrict__ w, int64_t rows, int cols,
                     const RowLanes<WHOLE> rl) {
  const int c = (int)blockIdx.x * 256 + rl.lane();  // the grid covers a row
  if (c >= cols) return;
  for (int64_t r = (int64_t)blockIdx.y * rl.per_wg() + rl.sub(); r < rows;
       r += (int64_t)gridDim.y * rl.per_wg()) {
    const float normed = through<DX>(F<DX>::up(x[r * sx + c]) * scale.at(r));
    out[r * so + c] = F<DO>::down(F<DW>::up(w[c]) * normed);
  }
}

// In place, x [n, heads, hd]: x = x * cos + rotate_half(x) * sin, rotate_half(x) =
// cat(-x2, x1), with cos / sin (fp32 [n, hd]) cast to the dtype first and every product
// and the sum rounded to it (HF's apply_rotary_pos_emb in the model dtype).
template <int DT>
__global__ void __launch_bounds__(256)
rope_kernel(typename F<DT>::S* __restrict__ x, int64_t sn, int64_t sh,
            const float* __restrict__ cs, const float* __restrict__ sn_, int64_t sc,
            int64_t n, int heads, int half) {
  const int64_t total = n * heads * half;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int d = (int)(i % half);
    const int64_t nh = i / half;
    const int h = (int)(nh % heads);
    const int64_t t = nh / heads;
    typename F<DT>::S* p = x + t * sn + h * sh;
    const float x1 = F<DT>::up(p[d]), x2 = F<DT>::up(p[d + half]);
    const float* c = cs + t * sc;
    const float* s = sn_ + t * sc;
    const float c1 = through<DT>(c[d]), c2 = through<DT>(c[d + half]);
    const float s1 = through<DT>(s[d]), s2 = through<DT>(s[d + half]);
    const float o1 = through<DT>(x1 * c1) + through<DT>(-x2 * s1);
    const float o2 = through<DT>(x2 * c2) + through<DT>(x1 * s2);
    p[d] = F<DT>::down(o1);
    p[d + half] = F<DT>::down(o2);
  }
}

// out = DT( f32(DT( g / (1 + exp(-g)) )) * u ): PyTorch's F.silu(gate) * up (SiLU in
// fp32 with the library exp and IEEE division, rounded, then the rounded product).
template <int DT>
__global__ void __launch_bounds__(256)
silu_mul_kernel(typename F<DT>::S* __restrict__ out, const typename F<DT>::S* __restrict__ g,
                const typename F<DT>::S* __restrict__ u, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const float gf = F<DT>::up(g[i]);
    const float silu = through<DT>(gf / (1.0f + expf(-gf)));
    out[i] = F<DT>::down(silu * F<DT>::up(u[i]));
  }
}

// The same three operations, 16 bytes per access (x, weight and output of one dtype for
// the RMSNorm tail; the launchers take these when pointers, strides and widths allow).
// Each element goes through exactly the scalar kernels' operations.
// One workgroup per row at a time; its first wave computes the row's scale (fp64: once per
// workgroup, not per thread) while the row's first loads are in flight.
template <int DT>
__global__ void __launch_bounds__(256)
rms_norm_tail_vec_kernel(typename F<DT>::S* __restrict__ out, int64_t so,
                         const typename F<DT>::S* __restrict__ x, int64_t sx,
                         const RowScale scale, const typename F<DT>::S* __restrict__ w,
                         int64_t rows, int cvec) {
  constexpr int V = VN<DT>;
  __shared__ float inv_s;
  for (int64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    int c = threadIdx.x;
    float xf[V], wf[V], o[V];
    if (c < cvec) {
      load16<DT>(x + r * sx + (int64_t)c * V, xf);
      load16<DT>(w + (int64_t)c * V, wf);
    }
    if (threadIdx.x < 64) {
      const float inv = scale.at(r);
      if (threadIdx.x == 0) inv_s = inv;
    }
    __syncthreads();
    const float inv = inv_s;
    __syncthreads();  // the next row's scale may be written
    while (c < cvec) {
#pragma unroll
      for (int j = 0; j < V; ++j) o[j] = xf[j] * inv;
      round_all<DT, V>(o);
#pragma unroll
      for (int j = 0; j < V; ++j) o[j] = wf[j] * o[j];
      store16<DT>(out + r * so + (int64_t)c * V, o);
      c += blockDim.x;
      if (c < cvec) {
        load16<DT>(x + r * sx + (int64_t)c * V, xf);
        load16<DT>(w + (int64_t)c * V, wf);
      }
    }
  }
}

// The same for rows of at most 64 vectors, several per workgroup: a row's threads lie in one
// wave, and each computes the scale itself.
template <int DT>
__global__ void __launch_bounds__(256)
rms_norm_tail_short_kernel(typename F<DT>::S* __restrict__ out, int64_t so,
                           const typename F<DT>::S* __restrict__ x, int64_t sx,
                           const RowScale scale, const typename F<DT>::S* __restrict__ w,
                           int64_t rows, int cvec, const RowLanes<false> rl) {
  constexpr int V = VN<DT>;
  const int c = rl.lane();
  if (c >= cvec) return;
  float wf[V];
  load16<DT>(w + (int64_t)c * V, wf);
  for (int64_t r = (int64_t)blockIdx.x * rl.per_wg() + rl.sub(); r < rows;
       r += (int64_t)gridDim.x * rl.per_wg()) {
    float o[V];
    load16<DT>(x + r * sx + (int64_t)c * V, o);
    const float inv = scale.at(r);
#pragma unroll
    for (int j = 0; j < V; ++j) o[j] *= inv;
    round_all<DT, V>(o);
#pragma unroll
    for (int j = 0; j < V; ++j) o[j] *= wf[j];
    store16<DT>(out + r * so + (int64_t)c * V, o);
  }
}

// sq[r, c] = f32(x[r, c])^2, sq contiguous: what PyTorch's x.float().pow(2) holds, in one pass
// (2,168 x 4,096 bf16: 8.9 us against 10.0 + 10.7 for the two).
template <int DT, bool WHOLE>
__global__ void __launch_bounds__(256)
square_kernel(float* __restrict__ sq, const typename F<DT>::S* __restrict__ x, int64_t sx,
              int64_t rows, int cols, const RowLanes<WHOLE> rl) {
  const int c = (int)blockIdx.x * 256 + rl.lane();  // the grid covers a row
  if (c >= cols) return;
  for (int64_t r = (int64_t)blockIdx.y * rl.per_wg() + rl.sub(); r < rows;
       r += (int64_t)gridDim.y * rl.per_wg()) {
    const float v = F<DT>::up(x[r * sx + c]);
    sq[r * cols + c] = v * v;
  }
}
// Four elements per access, so the fp32 stores of a wave are one contiguous piece.
template <int DT, bool WHOLE>
__global__ void __launch_bounds__(256)
square_vec_kernel(float* __restrict__ sq, const typename F<DT>::S* __restrict__ x, int64_t sx,
                  int64_t rows, int cvec, const RowLanes<WHOLE> rl) {
  const int c = (int)blockIdx.x * 256 + rl.lane();  // the grid covers a row
  if (c >= cvec) return;
  for (int64_t r = (int64_t)blockIdx.y * rl.per_wg() + rl.sub(); r < rows;
       r += (int64_t)gridDim.y * rl.per_wg()) {
    typename F<DT>::S v[4];
    const typename F<DT>::S* p = x + r * sx + (int64_t)c * 4;
    if constexpr (DT == PKV_F32) *reinterpret_cast<float4*>(v) = *reinterpret_cast<const float4*>(p);
    else *reinterpret_cast<uint2*>(v) = *reinterpret_cast<const uint2*>(p);
    float f[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) f[j] = F<DT>::up(v[j]) * F<DT>::up(v[j]);
    reinterpret_cast<float4*>(sq + r * cvec * 4)[c] = make_float4(f[0], f[1], f[2], f[3]);
  }
}

// A thread turns the same 2 x 16 bytes of HPT heads of one token, whose cos and sin it loads
// and rounds once; a workgroup holds per_wg tokens of `items` threads each (or one token,
// looped over, where a token has more items than threads). Index arithmetic is 32-bit but for
// the row addresses (it was three 64-bit divisions per 32 bytes). Bound by memory: 2,168 tokens,
// hd 128, bf16, 32 heads 14.6 -> 10.2 us (36 MB there and back), 8 heads 4.9 -> 4.5.
template <int DT, int HPT>
__global__ void __launch_bounds__(256)
rope_vec_kernel(typename F<DT>::S* __restrict__ x, int64_t sn, int64_t sh,
                const float* __restrict__ cs, const float* __restrict__ sn_, int64_t sc,
                int64_t n, int heads, int half, int items, int per_wg) {
  constexpr int V = VN<DT>;
  const int hv = half / V;
  const int sub = (int)threadIdx.x / items;  // 0 where a token fills the workgroup
  if (sub >= per_wg) return;
  for (int64_t t = (int64_t)blockIdx.x * per_wg + sub; t < n; t += (int64_t)gridDim.x * per_wg) {
    for (int i = (int)threadIdx.x - sub * items; i < items; i += 256) {
      const int hg = i / hv, d = (i - hg * hv) * V, h0 = hg * HPT;
      typename F<DT>::S* p = x + t * sn + h0 * sh + d;
      float x1[HPT][V], x2[HPT][V], c1[V], c2[V], s1[V], s2[V];
#pragma unroll
      for (int k = 0; k < HPT; ++k)
        if (h0 + k < heads) {
          load16<DT>(p + k * sh, x1[k]);
          load16<DT>(p + k * sh + half, x2[k]);
        }
      load_f32<V>(cs + t * sc + d, c1);
      load_f32<V>(cs + t * sc + d + half, c2);
      load_f32<V>(sn_ + t * sc + d, s1);
      load_f32<V>(sn_ + t * sc + d + half, s2);
      round_all<DT, V>(c1);
      round_all<DT, V>(c2);
      round_all<DT, V>(s1);
      round_all<DT, V>(s2);
#pragma unroll
      for (int k = 0; k < HPT; ++k)
        if (h0 + k < heads) {
          float a1[V], b1[V], a2[V], b2[V];
#pragma unroll
          for (int j = 0; j < V; ++j) {
            a1[j] = x1[k][j] * c1[j], b1[j] = -x2[k][j] * s1[j];
            a2[j] = x2[k][j] * c2[j], b2[j] = x1[k][j] * s2[j];
          }
          round_all<DT, V>(a1);
          round_all<DT, V>(b1);
          round_all<DT, V>(a2);
          round_all<DT, V>(b2);
#pragma unroll
          for (int j = 0; j < V; ++j) a1[j] += b1[j], a2[j] += b2[j];
          store16<DT>(p + k * sh, a1);
          store16<DT>(p + k * sh + half, a2);
        }
    }
  }
}

template <int DT, bool NT>
__global__ void __launch_bounds__(256)
silu_mul_vec_kernel(typename F<DT>::S* __restrict__ out, const typename F<DT>::S* __restrict__ g,
                    const typename F<DT>::S* __restrict__ u, int64_t nvec) {
  constexpr int V = VN<DT>;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nvec;
       i += (int64_t)gridDim.x * blockDim.x) {
    float gf[V], uf[V], o[V];
    load16<DT, NT>(g + i * V, gf);
    load16<DT, NT>(u + i * V, uf);
#pragma unroll
    for (int j = 0; j < V; ++j) o[j] = gf[j] / (1.0f + expf(-gf[j]));
    round_all<DT, V>(o);
#pragma unroll
    for (int j = 0; j < V; ++j) o[j] *= uf[j];
    store16<DT, NT>(out + i * V, o);
  }
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

bool valid(int dt) { return dt == PKV_F32 || dt == PKV_F16 || dt == PKV_BF16; }

// The dtype PyTorch promotes x (DX) and w (DW) to: equal dtypes stay, every mixed pair
// of the three floating types promotes to fp32.
int promoted(int dx, int dw) { return dx == dw ? dx : PKV_F32; }

unsigned blocks_for(int64_t n) {
  int64_t b = (n + 255) / 256;
  return (unsigned)(b < 1 ? 1 : (b > 8192 ? 8192 : b));
}

// Workgroups for kernels that loop over rows, one row (or packet of tokens) per workgroup at a
// time: HIP launches fewer than 2^32 threads along x.
unsigned row_grid(int64_t n) { return (unsigned)(n < (1 << 20) ? n : (1 << 20)); }

// Launch f's kernel<WHOLE> over rows of n: x workgroups along a row, y along the rows (the
// kernels loop over what is left).
template <class L> hipError_t launch_rows(int n, int64_t rows, const L& f) {
  if (n > 128) {
    f.template run<true>(dim3((unsigned)(((int64_t)n + 255) / 256), (unsigned)(rows < 65535 ? rows : 65535)),
                         RowLanes<true>(n));
  } else {
    const RowLanes<false> rl(n);
    const int64_t gy = (rows + rl.per_wg() - 1) / rl.per_wg();
    f.template run<false>(dim3(1, (unsigned)(gy < 65535 ? gy : 65535)), rl);
  }
  return hipGetLastError();
}
template <int DX, int DW, int DO> struct RmsScalar {
  void* out;
  int64_t so;
  const void* x;
  int64_t sx;
  const RowScale& inv;
  const void* w;
  int64_t rows;
  int cols;
  hipStream_t st;
  template <bool WHOLE> void run(dim3 grid, const RowLanes<WHOLE>& rl) const {
    hipLaunchKernelGGL((rms_norm_tail_kernel<DX, DW, DO, WHOLE>), grid, dim3(256), 0, st,
                       (typename F<DO>::S*)out, so, (const typename F<DX>::S*)x, sx, inv,
                       (const typename F<DW>::S*)w, rows, cols, rl);
  }
};
template <int DT> struct Square {
  float* sq;
  const void* x;
  int64_t sx, rows;
  int n;
  bool vec;
  hipStream_t st;
  template <bool WHOLE> void run(dim3 grid, const RowLanes<WHOLE>& rl) const {
    if (vec)
      hipLaunchKernelGGL((square_vec_kernel<DT, WHOLE>), grid, dim3(256), 0, st, sq,
                         (const typename F<DT>::S*)x, sx, rows, n, rl);
    else
      hipLaunchKernelGGL((square_kernel<DT, WHOLE>), grid, dim3(256), 0, st, sq,
                         (const typename F<DT>::S*)x, sx, rows, n, rl);
  }
};

template <int DX, int DW>
hipError_t launch_rms(void* out, int64_t so, const void* x, int64_t sx, const RowScale& inv,
                      const void* w, int64_t rows, int cols, hipStream_t st) {
  constexpr int DO = DX == DW ? DX : PKV_F32;
  if constexpr (DX == DW) {  // one dtype (the models' case): 16-byte accesses
    constexpr int V = VN<DX>;
    if (cols % V == 0 && sx % V == 0 && so % V == 0 && aligned16(out) && aligned16(x) &&
        aligned16(w)) {
      const int cvec = cols / V;
      const RowLanes<false> rl(cvec);
      if (cvec <= 64)
        hipLaunchKernelGGL((rms_norm_tail_short_kernel<DX>),
                           dim3(row_grid((rows + rl.per_wg() - 1) / rl.per_wg())), dim3(256), 0, st,
                           (typename F<DX>::S*)out, so, (const typename F<DX>::S*)x, sx, inv,
                           (const typename F<DX>::S*)w, rows, cvec, rl);
      else
        hipLaunchKernelGGL((rms_norm_tail_vec_kernel<DX>), dim3(row_grid(rows)), dim3(256), 0, st,
                           (typename F<DX>::S*)out, so, (const typename F<DX>::S*)x, sx, inv,
                           (const typename F<DX>::S*)w, rows, cvec);
      return hipGetLastError();
    }
  }
  return launch_rows(cols, rows, RmsScalar<DX, DW, DO>{out, so, x, sx, inv, w, rows, cols, st});
}

template <int DX>
hipError_t rms_by_w(int dw, void* out, int64_t so, const void* x, int64_t sx, const RowScale& inv,
                    const void* w, int64_t rows, int cols, hipStream_t st) {
  switch (dw) {
    case PKV_F32: return launch_rms<DX, PKV_F32>(out, so, x, sx, inv, w, rows, cols, st);
    case PKV_F16: return launch_rms<DX, PKV_F16>(out, so, x, sx, inv, w, rows, cols, st);
    default: return launch_rms<DX, PKV_BF16>(out, so, x, sx, inv, w, rows, cols, st);
  }
}

// Streaming accesses where the output alone is larger than the L2s (8 x 4 MB), so that the next
// kernel would not find it there either: 2,168 x 14,336 bf16 31.1 us against 34.7-36.9 (186 MB,
// 6.0 TB/s); streaming loads alone 35.2-36.7.
constexpr int64_t kStreamBytes = 32 << 20;
template <int DT>
hipError_t launch_silu(void* out, const void* g, const void* u, int64_t nvec, hipStream_t st) {
  using S = typename F<DT>::S;
  const unsigned nb = blocks_for(nvec);
  if (nvec * 16 >= kStreamBytes)
    hipLaunchKernelGGL((silu_mul_vec_kernel<DT, true>), dim3(nb), dim3(256), 0, st, (S*)out,
                       (const S*)g, (const S*)u, nvec);
  else
    hipLaunchKernelGGL((silu_mul_vec_kernel<DT, false>), dim3(nb), dim3(256), 0, st, (S*)out,
                       (const S*)g, (const S*)u, nvec);
  return hipGetLastError();
}

// Heads per thread of the vector RoPE: 4 once that leaves at least 128 Ki threads (two waves per
// SIMD of 256 CUs), else 1 (more threads in flight).
template <int DT, int HPT>
hipError_t launch_rope_hpt(void* x, int64_t sn, int64_t sh, const float* cs, const float* sn_,
                           int64_t sc, int64_t n, int heads, int half, hipStream_t st) {
  const int64_t items = (int64_t)((heads + HPT - 1) / HPT) * (half / VN<DT>);
  if (items > 0x7FFFFFFF) return hipErrorInvalidValue;
  const int per = items < 256 ? (int)(256 / items) : 1;
  const int64_t wgs = (n + per - 1) / per;
  hipLaunchKernelGGL((rope_vec_kernel<DT, HPT>), dim3(row_grid(wgs)),
                     dim3(256), 0, st, (typename F<DT>::S*)x, sn, sh, cs, sn_, sc, n, heads, half,
                     (int)items, per);
  return hipGetLastError();
}
template <int DT>
hipError_t launch_rope(void* x, int64_t sn, int64_t sh, const float* cs, const float* sn_,
                       int64_t sc, int64_t n, int heads, int half, hipStream_t st) {
  if (n * heads * (half / VN<DT>) >= (int64_t)4 << 17)
    return launch_rope_hpt<DT, 4>(x, sn, sh, cs, sn_, sc, n, heads, half, st);
  return launch_rope_hpt<DT, 1>(x, sn, sh, cs, sn_, sc, n, heads, half, st);
}

template <int DT>
hipError_t launch_square(float* sq, const void* x, int64_t sx, int64_t rows, int cols,
                         hipStream_t st) {
  const bool vec = cols % 4 == 0 && sx % 4 == 0 && aligned16(sq) && aligned16(x);
  const int n = vec ? cols / 4 : cols;
  return launch_rows(n, rows, Square<DT>{sq, x, sx, rows, n, vec, st});
}

int rms_norm(void* out, int out_dtype, int64_t out_stride_row, const void* x, int x_dtype,
             int64_t x_stride_row, const RowScale& inv_rms, const void* weight, int w_dtype,
             int64_t rows, int64_t cols, void* stream) {
  if (!valid(x_dtype) || !valid(w_dtype) || out_dtype != promoted(x_dtype, w_dtype))
    return PKV_E_DTYPE;
  if (rows < 0 || cols < 0 || cols > (1 << 30)) return PKV_E_SHAPE;
  if (rows == 0 || cols == 0) return 0;
  if (!out || !x || !inv_rms.v || !weight) return PKV_E_NULL;
  hipStream_t st = (hipStream_t)stream;
  const int c = (int)cols;
  switch (x_dtype) {
    case PKV_F32:
      return (int)rms_by_w<PKV_F32>(w_dtype, out, out_stride_row, x, x_stride_row, inv_rms,
                                    weight, rows, c, st);
    case PKV_F16:
      return (int)rms_by_w<PKV_F16>(w_dtype, out, out_stride_row, x, x_stride_row, inv_rms,
                                    weight, rows, c, st);
    default:
      return (int)rms_by_w<PKV_BF16>(w_dtype, out, out_stride_row, x, x_stride_row, inv_rms,
                                     weight, rows, c, st);
  }
}

}  // namespace

extern "C" {

int pkv_rms_norm(void* out, int out_dtype, int64_t out_stride_row, const void* x, int x_dtype,
                 int64_t x_stride_row, const float* inv_rms, const void* weight, int w_dtype,
                 int64_t rows, int64_t cols, void* stream) {
  return rms_norm(out, out_dtype, out_stride_row, x, x_dtype, x_stride_row,
                  RowScale{inv_rms, 0.f, false}, weight, w_dtype, rows, cols, stream);
}

int pkv_rms_norm_mean(void* out, int out_dtype, int64_t out_stride_row, const void* x, int x_dtype,
                      int64_t x_stride_row, const float* mean, float eps, const void* weight,
                      int w_dtype, int64_t rows, int64_t cols, void* stream) {
  return rms_norm(out, out_dtype, out_stride_row, x, x_dtype, x_stride_row,
                  RowScale{mean, eps, true}, weight, w_dtype, rows, cols, stream);
}

int pkv_square(float* out, const void* x, int dtype, int64_t x_stride_row, int64_t rows,
               int64_t cols, void* stream) {
  if (!valid(dtype)) return PKV_E_DTYPE;
  if (rows < 0 || cols < 0 || cols > (1 << 30)) return PKV_E_SHAPE;
  if (rows == 0 || cols == 0) return 0;
  if (!out || !x) return PKV_E_NULL;
  hipStream_t st = (hipStream_t)stream;
  switch (dtype) {
    case PKV_F32: return (int)launch_square<PKV_F32>(out, x, x_stride_row, rows, (int)cols, st);
    case PKV_F16: return (int)launch_square<PKV_F16>(out, x, x_stride_row, rows, (int)cols, st);
    default: return (int)launch_square<PKV_BF16>(out, x, x_stride_row, rows, (int)cols, st);
  }
}

int pkv_rope(void* x, int dtype, int64_t stride_tok, int64_t stride_head, const float* cos,
             const float* sin, int64_t cs_stride_tok, int64_t n_tokens, int32_t heads,
             int32_t head_dim, void* stream) {
  if (!valid(dtype)) return PKV_E_DTYPE;
  if (n_tokens < 0 || heads < 0 || head_dim < 0 || head_dim % 2) return PKV_E_SHAPE;
  if (n_tokens == 0 || heads == 0 || head_dim == 0) return 0;
  if (!x || !cos || !sin) return PKV_E_NULL;
  hipStream_t st = (hipStream_t)stream;
  const int half = head_dim / 2;
  const int v = dtype == PKV_F32 ? 4 : 8;  // elements per 16-byte access
  if (half % v == 0 && stride_tok % v == 0 && stride_head % v == 0 && cs_stride_tok % 4 == 0 &&
      aligned16(x) && aligned16(cos) && aligned16(sin)) {
    switch (dtype) {
      case PKV_F32:
        return (int)launch_rope<PKV_F32>(x, stride_tok, stride_head, cos, sin, cs_stride_tok,
                                         n_tokens, heads, half, st);
      case PKV_F16:
        return (int)launch_rope<PKV_F16>(x, stride_tok, stride_head, cos, sin, cs_stride_tok,
                                         n_tokens, heads, half, st);
      default:
        return (int)launch_rope<PKV_BF16>(x, stride_tok, stride_head, cos, sin, cs_stride_tok,
                                          n_tokens, heads, half, st);
    }
  }
  const unsigned nb = blocks_for(n_tokens * heads * half);
  switch (dtype) {
    case PKV_F32:
      hipLaunchKernelGGL(rope_kernel<PKV_F32>, dim3(nb), dim3(256), 0, st, (float*)x,
                         stride_tok, stride_head, cos, sin, cs_stride_tok, n_tokens, heads, half);
      break;
    case PKV_F16:
      hipLaunchKernelGGL(rope_kernel<PKV_F16>, dim3(nb), dim3(256), 0, st, (uint16_t*)x,
                         stride_tok, stride_head, cos, sin, cs_stride_tok, n_tokens, heads, half);
      break;
    default:
      hipLaunchKernelGGL(rope_kernel<PKV_BF16>, dim3(nb), dim3(256), 0, st, (uint16_t*)x,
                         stride_tok, stride_head, cos, sin, cs_stride_tok, n_tokens, heads, half);
  }
  return (int)hipGetLastError();
}

int pkv_silu_mul(void* out, const void* gate, const void* up, int dtype, int64_t n,
                 void* stream) {
  if (!valid(dtype)) return PKV_E_DTYPE;
  if (n < 0) return PKV_E_SHAPE;
  if (n == 0) return 0;
  if (!out || !gate || !up) return PKV_E_NULL;
  hipStream_t st = (hipStream_t)stream;
  const int v = dtype == PKV_F32 ? 4 : 8;  // elements per 16-byte access
  if (n % v == 0 && aligned16(out) && aligned16(gate) && aligned16(up)) {
    switch (dtype) {
      case PKV_F32: return (int)launch_silu<PKV_F32>(out, gate, up, n / v, st);
      case PKV_F16: return (int)launch_silu<PKV_F16>(out, gate, up, n / v, st);
      default: return (int)launch_silu<PKV_BF16>(out, gate, up, n / v, st);
    }
  }
  const unsigned nb = blocks_for(n);
  switch (dtype) {
    case PKV_F32:
      hipLaunchKernelGGL(silu_mul_kernel<PKV_F32>, dim3(nb), dim3(256), 0, st, (float*)out,
                         (const float*)gate, (const float*)up, n);
      break;
    case PKV_F16:
      hipLaunchKernelGGL(silu_mul_kernel<PKV_F16>, dim3(nb), dim3(256), 0, st,
                         (uint16_t*)out, (const uint16_t*)gate, (const uint16_t*)up, n);
      break;
    default:
      hipLaunchKernelGGL(silu_mul_kernel<PKV_BF16>, dim3(nb), dim3(256), 0, st,
                         (uint16_t*)out, (const uint16_t*)gate, (const uint16_t*)up, n);
  }
  return (int)hipGetLastError();
}

}  // extern "C"
