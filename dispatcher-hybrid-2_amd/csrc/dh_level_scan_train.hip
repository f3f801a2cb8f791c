// The level scan with its gradient, for training, gfx950.
//
// Forward (reference dispatcher_hybrid/modeling_dispatcher.py:86-88, 111-121), per (b, head, column):
//   m = [t >= 2^l] mask[b,t,l];  a = sigmoid(pre_i) m;  f = sigmoid(pre_f) m + 1 - m;  r = sigmoid(pre_r)
//   V_{l+1}[t] = f[t,l] V_l[t] + a[t,l] r[t-2^l,l] V_l[t-2^l]
// Backward, from G_n = dV_n down, s = t - 2^l:
//   q[t] = sum_c G[t,c] V_l[s,c]     dpre_i[t] = q r[s] m si (1 - si)     dpre_r[s] = q a[t] r[s] (1 - r[s])
//                                    dpre_f[t] = (sum_c G[t,c] V_l[t,c]) m sf (1 - sf)
//   G_l[t] = f[t] G_{l+1}[t] + a[t+2^l] r[t] G_{l+1}[t+2^l]
// The states V_1 .. V_{n-1} are kept from the forward in the model's dtype; sums, gates and the states inside a launch are
// fp32.
//
// Work decomposition: a wave is the 64 columns of one head, a position is one register, so a level is register arithmetic
// with the two gate values of a position broadcast from a lane (lane = position there) by v_readlane: no exchange through
// LDS and no barrier. Two launches per direction cover the levels, because a wave then holds every source it needs:
//   local    levels 0 .. 5 (lags 1 .. 32): 64 positions of its own plus a halo of 63 (recomputed: a third more updates)
//   strided  levels 6 .. 11 (lags 64 .. 2048): the up to 64 positions t = c (mod 64), closed under these lags
// The sums over columns (64 lanes) of 64 positions at a time go through a transposing reduction, ~2 instructions a value.
// Bound: VALU (forward ~4 instructions per state element and level, backward ~11) beside the states' traffic, one write
// and one read of n_lv x (b, T, d). Measured on MI355X at d 1024, 12 levels, bf16 (us): b 4, T 4096 forward 65 + 50,
// backward 96 + 101; b 4, T 1024 25 + 14 and 35 + 22. The torch loop took ~300 launches, 6.2 ms and 2.2 ms.
#include "dh_common.h"

#include <utility>

namespace {

constexpr int kCols = 64;           // head width, one lane per column
constexpr int kLocal = 6;           // levels 0 .. 5
constexpr int kWavesS = 8;          // strided: residue classes (waves) per workgroup
constexpr int kMaxT = 4096, kMaxLv = 12;

template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

// one element per lane; an offset past the range reads 0 and stores nothing
template <typename T> struct Row;
template <> struct Row<bf16_t> {
  __device__ __forceinline__ static float load(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __uint_as_float((uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0) << 16);
  }
  __device__ __forceinline__ static void store(__amdgpu_buffer_rsrc_t r, uint32_t off, float v) {
    __builtin_amdgcn_raw_buffer_store_b16((short)f32_to_bf16(v), r, off, 0, 0);
  }
};
template <> struct Row<float> {
  __device__ __forceinline__ static float load(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
  }
  __device__ __forceinline__ static void store(__amdgpu_buffer_rsrc_t r, uint32_t off, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, v), r, off, 0, 0);
  }
};

// Byte offset of a row walk: advances by a uniform step, one VALU add per row (opaque to the compiler, which otherwise
// keeps every row's offset of every level in scalar registers and spills them). A descriptor's range ends with the last
// row, so rows past T and before 0 (a wrapped offset) are out of range by themselves.
struct Walk {
  uint32_t off;
  __device__ __forceinline__ Walk(int t, uint32_t rb, uint32_t cb) : off((uint32_t)t * rb + cb) {}
  __device__ __forceinline__ uint32_t next(uint32_t step) {
    const uint32_t o = off;
    off += step;
    asm volatile("" : "+v"(off));
    return o;
  }
};
// Pins an updated state where it is computed, with a scheduling fence every 8 positions: the broadcast gate values stay
// few in scalar registers (otherwise the updates sink to their next use and hundreds of them spill).
#define DH_PIN(v, j)               \
  do {                             \
    asm volatile("" : "+v"(v));    \
    if (((j) & 7) == 0) __builtin_amdgcn_sched_barrier(0); \
  } while (0)

__device__ __forceinline__ float lane_of(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// (u, v) -> sums over lane pairs 32 (16) apart: u's in the lower half (even 16-lane rows), v's in the upper (odd rows)
__device__ __forceinline__ float merge32(float u, float v) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(u), __float_as_uint(v), false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
__device__ __forceinline__ float merge16(float u, float v) {
  const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(u), __float_as_uint(v), false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
// the same inside 16-lane rows: lanes without `bit` get u's pair sums, lanes with it v's; CTRL pairs a lane with one that
// differs in `bit` (and possibly in lower bits, which later steps sum over)
template <int CTRL>
__device__ __forceinline__ float merge_dpp(float u, float v, bool bit) {
  const float keep = bit ? v : u, send = bit ? u : v;
  return keep + dpp_move<CTRL, 0xf>(send);
}

// lane i gets the sum over all lanes of p[i mod N] (p is consumed)
template <int N>
__device__ __forceinline__ float column_sums(float (&p)[N], int lane) {
  static_assert(N == 64 || N == 32 || N == 16, "");
  if constexpr (N == 64)
#pragma unroll
    for (int k = 0; k < 32; ++k) p[k] = merge32(p[k], p[k + 32]);
  if constexpr (N >= 32)
#pragma unroll
    for (int k = 0; k < 16; ++k) p[k] = merge16(p[k], p[k + 16]);
#pragma unroll
  for (int k = 0; k < 8; ++k) p[k] = merge_dpp<0x128>(p[k], p[k + 8], lane & 8);     // row_ror:8
#pragma unroll
  for (int k = 0; k < 4; ++k) p[k] = merge_dpp<0x141>(p[k], p[k + 4], lane & 4);     // row_half_mirror
#pragma unroll
  for (int k = 0; k < 2; ++k) p[k] = merge_dpp<0x4e>(p[k], p[k + 2], lane & 2);      // quad_perm(2,3,0,1)
  float s = merge_dpp<0xb1>(p[0], p[1], lane & 1);                                   // quad_perm(1,0,3,2)
  if constexpr (N == 16) s = merge16(s, s);
  if constexpr (N <= 32) s = merge32(s, s);
  return s;
}

struct Args {
  const void* pre[3];           // element [b,t,l,h] at b spb + h sph + l spl + t
  int64_t spb, spl, sph;
  const void* mask;             // nullable
  int64_t smb, smt, sml;
  const void* V0;
  int64_t svb, svt;
  void* Vs;                     // (n_lv - 1, b, T, d): the states entering levels 1 .. n_lv - 1
  void* out;                    // forward: the scanned state (b, T, d)
  const void* dV;               // backward: its gradient, rows of d at b sgb + t sgt
  int64_t sgb, sgt;
  void* mid;                    // backward: gradient of the state entering level 6 (b, T, d)
  void* dV0;                    // rows of d at b sob + t sot
  int64_t sob, sot;
  void* dpre[3];                // laid out as pre
  int b, T, H, n_lv;
};

template <typename T>
__device__ __forceinline__ float mask_of(const Args& a, int b, int t, int l) {
  return a.mask == nullptr
             ? 1.f
             : Elem<T>::load((const T*)a.mask + (int64_t)b * a.smb + (int64_t)t * a.smt + (int64_t)l * a.sml);
}

// descriptor of the 64 columns of head h of one batch row, rows `st` elements apart
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t head_rows(const void* base, int64_t row0, int64_t st, int h, int T_) {
  return buf_rsrc((const T*)base + row0 + (int64_t)h * kCols,
                  (uint32_t)(((int64_t)(T_ - 1) * st + kCols) * (int64_t)sizeof(T)));
}

// the state entering level l (l >= 1), or the output for l == n_lv
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t state_rows(const Args& a, int l, int b, int h) {
  const int64_t d = (int64_t)a.H * kCols, plane = (int64_t)a.b * a.T * d;
  if (l == a.n_lv) return head_rows<T>(a.out, (int64_t)b * a.T * d, d, h, a.T);
  return head_rows<T>((const T*)a.Vs + (int64_t)(l - 1) * plane, (int64_t)b * a.T * d, d, h, a.T);
}

// the gates' logistic function: fp32 as torch evaluates it (library exp, IEEE divide), as the states and gradients are kept in
// full; bf16 pre-activations by the hardware exp and reciprocal (1 ulp of fp32 each, far below their own rounding)
template <typename T>
__device__ __forceinline__ float gate_sigmoid(float x) {
  if constexpr (sizeof(T) == 4) return 1.0f / (1.0f + expf(-x));
  return dh_sigmoid(x);
}

struct Gate {
  float m, si, sf, r;           // r: the transmit gate at the source
  __device__ __forceinline__ float f() const { return __builtin_fmaf(sf, m, 1.f - m); }
  __device__ __forceinline__ float a() const { return si * m; }
};

// lane-wise gates of position t (any integer; outside [lag, T) the edge does not exist: m = 0)
template <typename T>
__device__ __forceinline__ Gate gate_at(const Args& a, int b, int h, int l, int t) {
  const int lag = 1 << l;
  const bool in = t >= lag && t < a.T;
  const int tc = in ? t : 0, ts = in ? t - lag : 0;
  const int64_t row = (int64_t)b * a.spb + (int64_t)h * a.sph + (int64_t)l * a.spl;
  Gate g;
  g.si = gate_sigmoid<T>(Elem<T>::load((const T*)a.pre[0] + row + tc));
  g.sf = gate_sigmoid<T>(Elem<T>::load((const T*)a.pre[1] + row + tc));
  g.r = gate_sigmoid<T>(Elem<T>::load((const T*)a.pre[2] + row + ts));
  g.m = in ? mask_of<T>(a, b, tc, l) : 0.f;
  return g;
}

// ---- local levels ------------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256, 2) void scan_local_fwd(Args a) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = blockIdx.y * 4 + wave, b = blockIdx.z, s0 = blockIdx.x * 64;
  if (h >= a.H) return;                                       // no barrier below
  const uint32_t rb = (uint32_t)(a.svt * (int64_t)sizeof(T)), cb = lane * (uint32_t)sizeof(T);
  const uint32_t ob = (uint32_t)(a.H * kCols * (int)sizeof(T));
  float V[128];                                               // position s0 - 64 + j
  {
    const __amdgpu_buffer_rsrc_t r = head_rows<T>(a.V0, (int64_t)b * a.svb, a.svt, h, a.T);
    Walk o(s0 - 63, rb, cb);
#pragma unroll
    for (int j = 1; j < 128; ++j) V[j] = Row<T>::load(r, o.next(rb));
    V[0] = 0.f;
  }
  static_for<kLocal>([&](auto lc) {
    constexpr int l = decltype(lc)::value, lag = 1 << l;
    constexpr int first = 64 - (64 - 2 * lag);                // the halo the later levels still read: 64 - sum of their lags
    if (l >= a.n_lv) return;                                  // uniform
    const Gate g0 = gate_at<T>(a, b, h, l, s0 - 64 + lane), g1 = gate_at<T>(a, b, h, l, s0 + lane);
    const float f0 = g0.f(), c0 = g0.a() * g0.r, f1 = g1.f(), c1 = g1.a() * g1.r;
#pragma unroll
    for (int j = 127; j >= first; --j) {
      const float f = lane_of(j < 64 ? f0 : f1, j & 63), c = lane_of(j < 64 ? c0 : c1, j & 63);
      V[j] = __builtin_fmaf(c, V[j - lag], f * V[j]);
      DH_PIN(V[j], j);
    }
    const __amdgpu_buffer_rsrc_t r = state_rows<T>(a, l + 1, b, h);
    Walk o(s0, ob, cb);
#pragma unroll
    for (int j = 0; j < 64; ++j) Row<T>::store(r, o.next(ob), V[64 + j]);
  });
}

template <typename T>
__global__ __launch_bounds__(256, 2) void scan_local_bwd(Args a) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = blockIdx.y * 4 + wave, b = blockIdx.z, s0 = blockIdx.x * 64;
  if (h >= a.H) return;                                       // no barrier below
  const int64_t d = (int64_t)a.H * kCols;
  const bool top = a.n_lv <= kLocal;                          // no strided level: the incoming gradient itself
  const int64_t gst = top ? a.sgt : d;
  const uint32_t gb = (uint32_t)(gst * (int64_t)sizeof(T)), vb0 = (uint32_t)(a.svt * (int64_t)sizeof(T));
  const uint32_t ob = (uint32_t)(d * (int64_t)sizeof(T)), cb = lane * (uint32_t)sizeof(T);
  float G[128];                                               // position s0 + j
  {
    const __amdgpu_buffer_rsrc_t r =
        head_rows<T>(top ? a.dV : a.mid, (int64_t)b * (top ? a.sgb : (int64_t)a.T * d), gst, h, a.T);
    Walk o(s0, gb, cb);
#pragma unroll
    for (int j = 0; j < 127; ++j) G[j] = Row<T>::load(r, o.next(gb));
    G[127] = 0.f;
  }
  static_for<kLocal>([&](auto lc) {
    constexpr int l = kLocal - 1 - decltype(lc)::value, lag = 1 << l;
    constexpr int last = 63 + lag;                            // G_l is needed on [0, 63 + sum of the lower lags]
    if (l >= a.n_lv) return;                                  // uniform
    const int t = s0 + lane;
    const Gate g0 = gate_at<T>(a, b, h, l, t), g1 = gate_at<T>(a, b, h, l, t + 64);
    const __amdgpu_buffer_rsrc_t rv =
        l == 0 ? head_rows<T>(a.V0, (int64_t)b * a.svb, a.svt, h, a.T) : state_rows<T>(a, l > 0 ? l : 1, b, h);
    const uint32_t vb = l == 0 ? vb0 : ob;
    float s[2];                                               // lanes 0-31: sums with V[t], 32-63: with V[t - lag]
#pragma unroll
    for (int ch = 0; ch < 2; ++ch) {
      float p[64];
      Walk od(s0 + 32 * ch, vb, cb), os(s0 + 32 * ch - lag, vb, cb);
#pragma unroll
      for (int k = 0; k < 32; ++k) {                          // (a destination past T has G = 0)
        p[k] = G[32 * ch + k] * Row<T>::load(rv, od.next(vb));
        p[32 + k] = G[32 * ch + k] * Row<T>::load(rv, os.next(vb));
      }
      s[ch] = column_sums<64>(p, lane);
    }
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(s[0]), __float_as_uint(s[1]), false, false);
    const float df = __uint_as_float(sw[0]), q = __uint_as_float(sw[1]);
    if (t < a.T) {
      const int64_t row = (int64_t)b * a.spb + (int64_t)h * a.sph + (int64_t)l * a.spl;
      Elem<T>::store((T*)a.dpre[0] + row + t, q * g0.r * g0.m * (g0.si * (1.f - g0.si)));
      Elem<T>::store((T*)a.dpre[1] + row + t, df * g0.m * (g0.sf * (1.f - g0.sf)));
      // the transmit gate's gradient belongs to the source; a source past the last destination gets zero
      if (t >= lag) Elem<T>::store((T*)a.dpre[2] + row + t - lag, q * g0.a() * (g0.r * (1.f - g0.r)));
      if (t + lag >= a.T) Elem<T>::store((T*)a.dpre[2] + row + t, 0.f);
    }
    const float f0 = g0.f(), c0 = g0.a() * g0.r, f1 = g1.f(), c1 = g1.a() * g1.r;
#pragma unroll
    for (int j = 0; j < last; ++j) {
      const int k = j + lag;                                  // the destination this position feeds
      const float f = lane_of(j < 64 ? f0 : f1, j & 63), c = lane_of(k < 64 ? c0 : c1, k & 63);
      G[j] = __builtin_fmaf(c, G[k], f * G[j]);
      DH_PIN(G[j], j);
    }
  });
  const __amdgpu_buffer_rsrc_t r = head_rows<T>(a.dV0, (int64_t)b * a.sob, a.sot, h, a.T);
  const uint32_t db = (uint32_t)(a.sot * (int64_t)sizeof(T));
  Walk o(s0, db, cb);
#pragma unroll
  for (int j = 0; j < 64; ++j) Row<T>::store(r, o.next(db), G[j]);
}

// ---- strided levels ----------------------------------------------------------------------------------------------
// A workgroup's 8 waves are the classes c0 .. c0 + 7 of one (b, head); their gates pass through LDS so global memory sees
// 8 consecutive positions per access: gl[x][m][j][w] is the gate x of level 6 + m at position c0 + w + 64 j.
template <typename T, int P>
struct GateTile {
  T v[3][kMaxLv - kLocal][P][kWavesS];
};

template <typename T, int P, bool STORE>
__device__ __forceinline__ void move_gates(const Args& a, GateTile<T, P>& gl, int b, int h, int c0) {
  constexpr int W16 = kWavesS * (int)sizeof(T) / 16;          // 16-byte words of 8 elements
  const int nl = a.n_lv - kLocal;
  for (int e = threadIdx.x; e < 3 * nl * P; e += 64 * kWavesS) {
    const int j = e % P, xm = e / P, x = xm / nl, m = xm - x * nl;
    const int t = c0 + 64 * j;
    const int64_t off = (int64_t)b * a.spb + (int64_t)h * a.sph + (int64_t)(kLocal + m) * a.spl + t;
    uint4* s = reinterpret_cast<uint4*>(&gl.v[x][m][j][0]);
    if constexpr (STORE) {
      uint4* g = reinterpret_cast<uint4*>((T*)(x == 0 ? a.dpre[0] : x == 1 ? a.dpre[1] : a.dpre[2]) + off);
      if (t < a.T)
#pragma unroll
        for (int i = 0; i < W16; ++i) g[i] = s[i];
    } else {
      const uint4* g = reinterpret_cast<const uint4*>((const T*)(x == 0 ? a.pre[0] : x == 1 ? a.pre[1] : a.pre[2]) + off);
#pragma unroll
      for (int i = 0; i < W16; ++i) s[i] = t < a.T ? g[i] : make_uint4(0, 0, 0, 0);
    }
  }
}

template <typename T, int P>
__device__ __forceinline__ Gate tile_gate(const Args& a, const GateTile<T, P>& gl, int b, int m, int c, int w, int lane) {
  const int lg = 1 << m, t = c + 64 * lane;                   // lag in units of 64 positions
  const bool in = lane < P && lane >= lg && t < a.T;
  const int j = in ? lane : 0, js = in ? lane - lg : 0;
  Gate g;
  g.si = gate_sigmoid<T>(Elem<T>::load(&gl.v[0][m][j][w]));
  g.sf = gate_sigmoid<T>(Elem<T>::load(&gl.v[1][m][j][w]));
  g.r = gate_sigmoid<T>(Elem<T>::load(&gl.v[2][m][js][w]));
  g.m = in ? mask_of<T>(a, b, t, kLocal + m) : 0.f;
  return g;
}

template <typename T, int P>
__global__ __launch_bounds__(64 * kWavesS, 2) void scan_strided_fwd(Args a) {
  __shared__ __align__(16) GateTile<T, P> gl;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c0 = blockIdx.x * kWavesS, h = blockIdx.y, b = blockIdx.z, c = c0 + w;
  const uint32_t ob = (uint32_t)(a.H * kCols * (int)sizeof(T)), cb = lane * (uint32_t)sizeof(T);
  float V[P];
  {
    const __amdgpu_buffer_rsrc_t r = state_rows<T>(a, kLocal, b, h);
    Walk o(c, ob, cb);
#pragma unroll
    for (int j = 0; j < P; ++j) V[j] = Row<T>::load(r, o.next(64 * ob));
  }
  move_gates<T, P, false>(a, gl, b, h, c0);
  __syncthreads();
  static_for<kMaxLv - kLocal>([&](auto mc) {
    constexpr int m = decltype(mc)::value, lg = 1 << m;
    if (kLocal + m >= a.n_lv) return;                         // uniform
    const Gate g = tile_gate<T, P>(a, gl, b, m, c, w, lane);
    const float fv = g.f(), cv = g.a() * g.r;
#pragma unroll
    for (int j = P - 1; j >= lg; --j) {
      V[j] = __builtin_fmaf(lane_of(cv, j), V[j - lg], lane_of(fv, j) * V[j]);
      DH_PIN(V[j], j);
    }
    const __amdgpu_buffer_rsrc_t r = state_rows<T>(a, kLocal + m + 1, b, h);
    Walk o(c, ob, cb);
#pragma unroll
    for (int j = 0; j < P; ++j) Row<T>::store(r, o.next(64 * ob), V[j]);
  });
}

template <typename T, int P>
__global__ __launch_bounds__(64 * kWavesS, 2) void scan_strided_bwd(Args a) {
  __shared__ __align__(16) GateTile<T, P> gl;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c0 = blockIdx.x * kWavesS, h = blockIdx.y, b = blockIdx.z, c = c0 + w;
  const int64_t d = (int64_t)a.H * kCols;
  const uint32_t ob = (uint32_t)(d * (int64_t)sizeof(T)), gb = (uint32_t)(a.sgt * (int64_t)sizeof(T));
  const uint32_t cb = lane * (uint32_t)sizeof(T);
  float G[P];
  {
    const __amdgpu_buffer_rsrc_t r = head_rows<T>(a.dV, (int64_t)b * a.sgb, a.sgt, h, a.T);
    Walk o(c, gb, cb);
#pragma unroll
    for (int j = 0; j < P; ++j) G[j] = Row<T>::load(r, o.next(64 * gb));
  }
  move_gates<T, P, false>(a, gl, b, h, c0);
  __syncthreads();
  static_for<kMaxLv - kLocal>([&](auto mc) {
    constexpr int m = kMaxLv - kLocal - 1 - decltype(mc)::value, lg = 1 << m;
    if (kLocal + m >= a.n_lv) return;                         // uniform
    const Gate g = tile_gate<T, P>(a, gl, b, m, c, w, lane);
    const __amdgpu_buffer_rsrc_t r = state_rows<T>(a, kLocal + m, b, h);
    float V[P], p[P];
    Walk o(c, ob, cb);
#pragma unroll
    for (int j = 0; j < P; ++j) V[j] = Row<T>::load(r, o.next(64 * ob));
#pragma unroll
    for (int j = 0; j < P; ++j) p[j] = G[j] * V[j];
    const float df = column_sums<P>(p, lane);
#pragma unroll
    for (int j = 0; j < P; ++j) p[j] = j >= lg ? G[j] * V[j >= lg ? j - lg : 0] : 0.f;
    const float q = column_sums<P>(p, lane);
    // the gradients take the gates' place in the tile: this wave's column w of level m is read by no one else
    if (lane < P) {
      const int t = c + 64 * lane;
      Elem<T>::store(&gl.v[0][m][lane][w], q * g.r * g.m * (g.si * (1.f - g.si)));
      Elem<T>::store(&gl.v[1][m][lane][w], df * g.m * (g.sf * (1.f - g.sf)));
      if (lane >= lg && t < a.T) Elem<T>::store(&gl.v[2][m][lane - lg][w], q * g.a() * (g.r * (1.f - g.r)));
      if (t + 64 * lg >= a.T) Elem<T>::store(&gl.v[2][m][lane][w], 0.f);
    }
    const float fv = g.f(), cv = g.a() * g.r;
#pragma unroll
    for (int j = 0; j < P; ++j) {
      const float fg = lane_of(fv, j) * G[j];
      G[j] = j + lg < P ? __builtin_fmaf(lane_of(cv, j + lg < P ? j + lg : 0), G[j + lg < P ? j + lg : 0], fg) : fg;
      DH_PIN(G[j], j);
    }
  });
  {
    const __amdgpu_buffer_rsrc_t r = head_rows<T>(a.mid, (int64_t)b * a.T * d, d, h, a.T);
    Walk o(c, ob, cb);
#pragma unroll
    for (int j = 0; j < P; ++j) Row<T>::store(r, o.next(64 * ob), G[j]);
  }
  __syncthreads();
  move_gates<T, P, true>(a, gl, b, h, c0);
}

template <typename T>
void run_fwd(const Args& a, hipStream_t s) {
  scan_local_fwd<T><<<dim3((a.T + 63) / 64, (a.H + 3) / 4, a.b), 256, 0, s>>>(a);
  if (a.n_lv <= kLocal) return;
  const dim3 grid(64 / kWavesS, a.H, a.b), block(64 * kWavesS);
  if (a.T <= 1024) scan_strided_fwd<T, 16><<<grid, block, 0, s>>>(a);
  else if (a.T <= 2048) scan_strided_fwd<T, 32><<<grid, block, 0, s>>>(a);
  else scan_strided_fwd<T, 64><<<grid, block, 0, s>>>(a);
}

template <typename T>
void run_bwd(const Args& a, hipStream_t s) {
  if (a.n_lv > kLocal) {
    const dim3 grid(64 / kWavesS, a.H, a.b), block(64 * kWavesS);
    if (a.T <= 1024) scan_strided_bwd<T, 16><<<grid, block, 0, s>>>(a);
    else if (a.T <= 2048) scan_strided_bwd<T, 32><<<grid, block, 0, s>>>(a);
    else scan_strided_bwd<T, 64><<<grid, block, 0, s>>>(a);
  }
  scan_local_bwd<T><<<dim3((a.T + 63) / 64, (a.H + 3) / 4, a.b), 256, 0, s>>>(a);
}

bool aligned(const void* p, uintptr_t n) { return ((uintptr_t)p % n) == 0; }

int check_train(const char* who, int dtype, int64_t spb, int64_t spl, int64_t sph, int64_t svb, int64_t svt, int b, int T,
                int H, int hd, int n_lv) {
  DH_REQUIRE(dtype == DH_F32 || dtype == DH_BF16, DH_ERR_UNSUPPORTED_DTYPE, "%s: dtype %d", who, dtype);
  DH_REQUIRE(b >= 1 && b <= 65535 && T >= 1 && T <= kMaxT, DH_ERR_UNSUPPORTED_SHAPE, "%s: b=%d (1..65535) T=%d (1..%d)",
             who, b, T, kMaxT);
  DH_REQUIRE(H >= 1 && H <= 64 && hd == kCols, DH_ERR_UNSUPPORTED_SHAPE, "%s: H=%d (1..64) hd=%d (%d)", who, H, hd, kCols);
  // a level whose lag reaches past T has no edge; the strided launches hold T / 64 positions a class
  DH_REQUIRE(n_lv >= 1 && n_lv <= kMaxLv, DH_ERR_UNSUPPORTED_SHAPE, "%s: n_lv=%d (1..%d)", who, n_lv, kMaxLv);
  DH_REQUIRE(spl >= T && spl % 8 == 0 && sph % 8 == 0 && spb % 8 == 0, DH_ERR_INVALID_ARG,
             "%s: gate rows are contiguous along t, at least T long, and start on multiples of 8 elements", who);
  // (a tile's halo reaches up to 127 rows past either end of a batch row: those 32-bit offsets must not wrap into range)
  DH_REQUIRE(svt >= (int64_t)H * hd && svb >= 0 && (int64_t)(T + 128) * svt * 4 < ((int64_t)1 << 31), DH_ERR_INVALID_ARG,
             "%s: row stride %lld", who, (long long)svt);
  return DH_OK;
}

}  // namespace

extern "C" int dh_level_scan_train_fwd(int dtype, const void* pre_i, const void* pre_f, const void* pre_r,
                                       int64_t stride_pb, int64_t stride_pl, int64_t stride_ph, const void* mask,
                                       int64_t stride_mb, int64_t stride_mt, int64_t stride_ml, const void* V0,
                                       int64_t stride_vb, int64_t stride_vt, void* states, void* V, int b, int T, int H,
                                       int hd, int n_lv, void* stream) {
  const char* who = "dh_level_scan_train_fwd";
  const int st = check_train(who, dtype, stride_pb, stride_pl, stride_ph, stride_vb, stride_vt, b, T, H, hd, n_lv);
  if (st) return st;
  DH_REQUIRE(pre_i && pre_f && pre_r && V0 && V && (states || n_lv == 1), DH_ERR_INVALID_ARG, "%s: null pointer argument",
             who);
  DH_REQUIRE(aligned(pre_i, 16) && aligned(pre_f, 16) && aligned(pre_r, 16), DH_ERR_INVALID_ARG,
             "%s: the gates need 16-byte alignment", who);
  Args a{};
  a.pre[0] = pre_i;
  a.pre[1] = pre_f;
  a.pre[2] = pre_r;
  a.spb = stride_pb;
  a.spl = stride_pl;
  a.sph = stride_ph;
  a.mask = mask;
  a.smb = stride_mb;
  a.smt = stride_mt;
  a.sml = stride_ml;
  a.V0 = V0;
  a.svb = stride_vb;
  a.svt = stride_vt;
  a.Vs = states;
  a.out = V;
  a.b = b;
  a.T = T;
  a.H = H;
  a.n_lv = n_lv;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == DH_F32) run_fwd<float>(a, s);
  else run_fwd<bf16_t>(a, s);
  return dh_check_launch(who);
}

extern "C" int dh_level_scan_train_bwd(int dtype, const void* pre_i, const void* pre_f, const void* pre_r,
                                       int64_t stride_pb, int64_t stride_pl, int64_t stride_ph, const void* mask,
                                       int64_t stride_mb, int64_t stride_mt, int64_t stride_ml, const void* V0,
                                       int64_t stride_vb, int64_t stride_vt, const void* states, const void* dV,
                                       int64_t stride_gb, int64_t stride_gt, void* scratch, void* dV0,
                                       int64_t stride_ob, int64_t stride_ot, void* dpre_i, void* dpre_f, void* dpre_r, int b, int T, int H, int hd, int n_lv, void* stream) {
  const char* who = "dh_level_scan_train_bwd";
  int st = check_train(who, dtype, stride_pb, stride_pl, stride_ph, stride_vb, stride_vt, b, T, H, hd, n_lv);
  if (!st) st = check_train(who, dtype, stride_pb, stride_pl, stride_ph, stride_gb, stride_gt, b, T, H, hd, n_lv);
  if (!st) st = check_train(who, dtype, stride_pb, stride_pl, stride_ph, stride_ob, stride_ot, b, T, H, hd, n_lv);
  if (st) return st;
  DH_REQUIRE(pre_i && pre_f && pre_r && V0 && (states || n_lv == 1) && dV && dV0 && dpre_i && dpre_f && dpre_r &&
                 (scratch || n_lv <= kLocal),
             DH_ERR_INVALID_ARG, "%s: null pointer argument", who);
  DH_REQUIRE(aligned(pre_i, 16) && aligned(pre_f, 16) && aligned(pre_r, 16) && aligned(dpre_i, 16) && aligned(dpre_f, 16) &&
                 aligned(dpre_r, 16),
             DH_ERR_INVALID_ARG, "%s: the gates and their gradients need 16-byte alignment", who);
  Args a{};
  a.pre[0] = pre_i;
  a.pre[1] = pre_f;
  a.pre[2] = pre_r;
  a.spb = stride_pb;
  a.spl = stride_pl;
  a.sph = stride_ph;
  a.mask = mask;
  a.smb = stride_mb;
  a.smt = stride_mt;
  a.sml = stride_ml;
  a.V0 = V0;
  a.svb = stride_vb;
  a.svt = stride_vt;
  a.Vs = const_cast<void*>(states);
  a.dV = dV;
  a.sgb = stride_gb;
  a.sgt = stride_gt;
  a.mid = scratch;
  a.dV0 = dV0;
  a.sob = stride_ob;
  a.sot = stride_ot;
  a.dpre[0] = dpre_i;
  a.dpre[1] = dpre_f;
  a.dpre[2] = dpre_r;
  a.b = b;
  a.T = T;
  a.H = H;
  a.n_lv = n_lv;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == DH_F32) run_bwd<float>(a, s);
  else run_bwd<bf16_t>(a, s);
  return dh_check_launch(who);
}
