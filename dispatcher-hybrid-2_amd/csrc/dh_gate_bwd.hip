// Backward of the gate pre-activations on the matrix cores, gfx950.
//
// Semantics (reference dispatcher_hybrid/fused_gates.py:96-173), per level l (lag 2^l), head h, gate x:
//   ok[t,l]   = t >= 2^l && (mask == null || mask[b,t,l] > 0)
//   x[t,l,k]  = relu(round(A[t,k] + ok B[t-2^l,k])),  hid = round(x^2)         (the forward's rounding points)
//   dh[t,l,k] = sum_{x,h} dP_x[t,l,h] W_x[l,h,k]
//   dA[t,k]   = sum_l 2 x[t,l,k] dh[t,l,k]
//   dB[s,k]   = sum_l ok[s+2^l,l] 2 x[s+2^l,l,k] dh[s+2^l,l,k]                  (gathered at the source: no atomics)
//   dW_x[l,h,k] = sum_{b,t} dP_x[t,l,h] hid[t,l,k],   db_x[l,h] = sum_{b,t} dP_x[t,l,h]
//
// Four launches, all sums in fp32 and in a fixed order (the same inputs give the same bits):
//   gate_bwd_pack    the gradients dP, in whatever layout, into the two MFMA fragment orders below, and the masks into
//                    two 16-bit sets per position (one pass over dP; everything after reads 16 bytes per lane, linearly)
//   gate_bwd_ab      dA and dB: both contractions over the 3 H gate outputs, one operand resident
//   gate_bwd_w       dW and db: contractions over positions, split over row ranges
//   gate_bwd_reduce  the ranges' partial sums, added in order and rounded once to the gradients' dtype
//
// Measured on MI355X (16 heads, 12 levels, GH 1024; us): bf16 b 4, T 4096: pack 15 + ab 166 + w 93 + reduce 6, where the
// atomic kernel of dh_gate_preacts_bwd takes 8361; b 4, T 1024: 8 + 44 + 28 + 6 against 5115; fp32 b 1, T 777: 105
// against 3944.
#include "dh_common.h"

namespace {

typedef short v8i16 __attribute__((ext_vector_type(8)));
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

constexpr uint32_t kOob = 0x80000000u;   // a buffer offset past every descriptor's range: the load returns zeros

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ uint4 bld16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
__device__ __forceinline__ uint2 bld8(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}
__device__ __forceinline__ float bld4f(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
__device__ __forceinline__ uint32_t bld4(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  bf16x2_t v;
  v.x = (__bf16)lo;
  v.y = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, v);
}
// bf16-valued fp32 of an ordinary (not transcendental) VALU result: bf16(x) in the high half, bf16(0) in the low
__device__ __forceinline__ float round_hi(float x) {
  float r;
  asm("v_cvt_pk_bf16_f32 %0, 0, %1" : "=v"(r) : "v"(x));
  return r;
}

template <typename T> struct Lay;
// K: elements of one 16-byte piece; TB: positions of one dW block (one MFMA contraction, times 4 in fp32);
// NM: 16-row MFMA tiles of one 128-byte column tile
template <> struct Lay<bf16_t> { static constexpr int K = 8, KT = 64, NM = 4, TB = 32; };
template <> struct Lay<float> { static constexpr int K = 4, KT = 32, NM = 2, TB = 16; };

// ---- fragment orders of dP ---------------------------------------------------------------------------------------
// A pair p = (level l, group nt of 16 heads), p = l * NT + nt, NP = n_lv * NT.
// P1, contraction over the gates (gate_bwd_ab): for position t = 16 tile + r and heads 16 nt + 4 g .. + 3, index
//   ((b NP + p) NT16 + tile) 64 + 16 g + r; bf16: plane 0 holds {dP_i x4, dP_f x4} (16 bytes), plane 1 dP_r x4 (8 bytes);
//   fp32: planes of dP_i x4, dP_f x4, dP_r x4 (16 bytes each).
// P2, contraction over positions (gate_bwd_w): for gate x, head 16 nt + h and the K positions from TB blk + K g, index
//   (((b NP + p) 3 + x) NBK + blk) 64 + 16 g + h, 16 bytes.
// Heads >= H and positions >= T are zeros.
struct Dims {
  int b, T, GH, H, n_lv, NT, NP, NT16, NBK;
};

struct PackArgs {
  const void* dP[3];
  int64_t sb, st, sl, sh;
  const void* mask;
  int64_t smb, smt, sml;
  void* p1;
  uint4* p2;
  uint32_t* ok;
  bool wide;                    // dP rows contiguous along t, starting on 16-byte boundaries
  Dims d;
};

constexpr int kPackRows = 64;

template <typename T>
__global__ __launch_bounds__(256) void gate_bwd_pack(PackArgs a) {
  constexpr int RS = kPackRows + 16 / (int)sizeof(T);        // padded LDS row (elements), 16-byte units stay aligned
  extern __shared__ __align__(16) unsigned char raw[];
  T* tile = (T*)raw;                                         // [3 H][RS]
  const Dims& d = a.d;
  const int b = blockIdx.z, l = blockIdx.y, t0 = blockIdx.x * kPackRows, tid = threadIdx.x;
  __shared__ uint32_t part[4][kPackRows];
  if (l == 0) {
    // bit j: level j reaches t from t - 2^j (low half); level j carries t to t + 2^j (high half). A thread takes every
    // fourth level of a position and has its 8 mask values in flight together
    const int i = tid & (kPackRows - 1), t = t0 + i, q = tid / kPackRows;
    uint32_t bits = 0;
    float in[4], out[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = min(q + 4 * u, d.n_lv - 1);
      auto at = [&](int tt) {
        return a.mask == nullptr ? 1.f
                                 : Elem<T>::load((const T*)a.mask + (int64_t)b * a.smb + (int64_t)min(tt, d.T - 1) * a.smt +
                                                 (int64_t)j * a.sml);
      };
      in[u] = at(t);
      out[u] = at(t + (1 << j));
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = q + 4 * u;
      if (j >= d.n_lv) continue;
      if (t >= (1 << j) && in[u] > 0.f) bits |= 1u << j;
      if (t + (1 << j) < d.T && out[u] > 0.f) bits |= 1u << (16 + j);
    }
    part[q][i] = bits;
  }
  if (a.wide) {
    // rows contiguous along t and 16-byte aligned: a 16-byte piece per thread (with the mask loads above in flight together,
    // b 4, T 4096: 26 us with single elements -> 15)
    constexpr int V = 16 / (int)sizeof(T), CPR = kPackRows / V;
    for (int e = tid; e < 3 * d.H * CPR; e += 256) {
      const int row = e / CPR, i = (e % CPR) * V, t = t0 + i;            // row = x H + h
      const int x = row < d.H ? 0 : row < 2 * d.H ? 1 : 2, h = row - x * d.H;
      const T* p = (const T*)(x == 0 ? a.dP[0] : x == 1 ? a.dP[1] : a.dP[2]) + (int64_t)b * a.sb + (int64_t)l * a.sl +
                   (int64_t)h * a.sh + t;
      T v[V];
      if (t + V <= d.T) {
        const uint4 u = *reinterpret_cast<const uint4*>(p);
        __builtin_memcpy(v, &u, 16);
      } else {
#pragma unroll
        for (int k = 0; k < V; ++k) v[k] = t + k < d.T ? p[k] : (T)0;
      }
      uint4 u;
      __builtin_memcpy(&u, v, 16);
      *reinterpret_cast<uint4*>(&tile[row * RS + i]) = u;
    }
  } else {
    const int n = 3 * d.H * kPackRows;
    for (int e = tid; e < n; e += 256) {
      // consecutive threads follow the layout's unit stride: along t (head-major) or along h
      int x, h, i;
      if (a.st == 1) {
        i = e & (kPackRows - 1);
        const int q = e / kPackRows;
        x = q / d.H;
        h = q - x * d.H;
      } else {
        const int q = e / d.H;
        h = e - q * d.H;
        x = q / kPackRows;
        i = q & (kPackRows - 1);
      }
      const T* p = (const T*)(x == 0 ? a.dP[0] : x == 1 ? a.dP[1] : a.dP[2]);
      T v = 0;
      if (t0 + i < d.T) v = p[(int64_t)b * a.sb + (int64_t)(t0 + i) * a.st + (int64_t)l * a.sl + (int64_t)h * a.sh];
      tile[(x * d.H + h) * RS + i] = v;
    }
  }
  __syncthreads();
  if (l == 0 && tid < kPackRows && t0 + tid < d.T)
    a.ok[(int64_t)b * d.T + t0 + tid] = part[0][tid] | part[1][tid] | part[2][tid] | part[3][tid];
  for (int nt = 0; nt < d.NT; ++nt) {
    const int64_t pair = (int64_t)b * d.NP + l * d.NT + nt;
    {
      const int r = tid & 15, g = (tid >> 4) & 3, tl = tid >> 6, tg = (t0 >> 4) + tl;
      if (tg < d.NT16) {
        T v[3][4];
#pragma unroll
        for (int x = 0; x < 3; ++x)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int h = nt * 16 + 4 * g + e;
            v[x][e] = h < d.H ? tile[(x * d.H + h) * RS + tl * 16 + r] : (T)0;
          }
        const int64_t idx = (pair * d.NT16 + tg) * 64 + g * 16 + r;
        const int64_t plane = (int64_t)d.b * d.NP * d.NT16 * 64;
        if constexpr (sizeof(T) == 2) {
          uint4 u;
          uint2 w;
          __builtin_memcpy(&u.x, v[0], 8);
          __builtin_memcpy(&u.z, v[1], 8);
          __builtin_memcpy(&w, v[2], 8);
          ((uint4*)a.p1)[idx] = u;
          ((uint2*)((uint4*)a.p1 + plane))[idx] = w;
        } else {
#pragma unroll
          for (int x = 0; x < 3; ++x) {
            uint4 u;
            __builtin_memcpy(&u, v[x], 16);
            ((uint4*)a.p1)[x * plane + idx] = u;
          }
        }
      }
    }
    constexpr int TB = Lay<T>::TB, K = Lay<T>::K, NB = kPackRows / TB;
    for (int u = tid; u < 3 * NB * 64; u += 256) {
      const int x = u / (NB * 64), blk = (u >> 6) % NB, g = (u >> 4) & 3, hh = u & 15, h = nt * 16 + hh;
      const int bg = t0 / TB + blk;
      if (bg >= d.NBK) continue;
      uint4 v = make_uint4(0, 0, 0, 0);
      if (h < d.H) v = *reinterpret_cast<const uint4*>(&tile[(x * d.H + h) * RS + blk * TB + g * K]);
      a.p2[((pair * 3 + x) * d.NBK + bg) * 64 + g * 16 + hh] = v;
    }
  }
}

// ---- dA and dB ---------------------------------------------------------------------------------------------------
// One workgroup (8 waves) owns a 128-byte column tile (64 bf16 / 32 fp32 columns) and walks row tiles; blockIdx.z picks
// dA (own rows A, lagged rows B at t - 2^l) or dB (own rows B, lagged rows A at s + 2^l). The tile's transposed weights
// of kPairs (level, head group) pairs sit in LDS for the whole walk (72 KB: two workgroups per CU; no barrier between
// row tiles), so a wave is on its own: 16 rows, own operand in registers, per pair two 16-byte lagged pieces per lane
// and one dP fragment, both requested one pair ahead; dh^T = W^T dP^T on MFMA puts 4 consecutive columns of one row in
// a lane, the layout the pieces arrive in (piece g and 4 + g of the row), so dx needs no further moves.
// Bound: VALU, ~5 instructions per element and level (unpack, add, clamp, round, multiply-add) over two passes of
// rows x GH x levels elements, beside 8 ds_bpermute per 1024 elements.
struct AbArgs {
  const void* A;
  const void* B;
  int64_t sab, sat;
  const void* W[3];
  int64_t swl, swh;
  const void* p1;
  const uint32_t* ok;
  void* dA;                     // rows of GH at b sgb + t sgt, both
  void* dB;
  int64_t sgb, sgt;
  Dims d;
};

constexpr int kPairs = 12;
constexpr int kAbThreads = 512;

template <typename T, typename OT>
__global__ __launch_bounds__(kAbThreads, 4) void gate_bwd_ab(AbArgs a) {
  typedef Lay<T> Y;
  constexpr int NM = Y::NM, K = Y::K;
  constexpr int ROWS = NM * 16;                              // LDS weight rows of a pair, row q = 16 m + r
  __shared__ __align__(16) unsigned char wl[kPairs * 6144];
  const Dims& d = a.d;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int k0 = blockIdx.x * Y::KT;
  const bool is_b = blockIdx.z != 0;
  const int crow = lane >> 2, cpiece = lane & 3;             // coalesced load: piece lane & 3 of row lane >> 2
  const int bperm = 4 * (4 * r + g);
  auto to_mfma = [&](const uint4& v) {
    return make_uint4((uint32_t)__builtin_amdgcn_ds_bpermute(bperm, (int)v.x),
                      (uint32_t)__builtin_amdgcn_ds_bpermute(bperm, (int)v.y),
                      (uint32_t)__builtin_amdgcn_ds_bpermute(bperm, (int)v.z),
                      (uint32_t)__builtin_amdgcn_ds_bpermute(bperm, (int)v.w));
  };
  // LDS weights, W^T rows: bf16: 64-byte rows {i x4, f x4} per head group g, then 32-byte rows r x4; fp32: three planes
  // of 64-byte rows. The 16-byte (8-byte) chunk g of row q is kept at g ^ ((q >> 1) & 3) (g ^ ((q >> 2) & 3)): the 16
  // rows a fragment read takes then fall on distinct banks.
  auto w_off = [&](int pr, int q, int x, int gg) -> int {
    if constexpr (sizeof(T) == 2)
      return x < 2 ? pr * 6144 + q * 64 + ((gg ^ ((q >> 1) & 3)) * 16) + x * 8
                   : pr * 6144 + 4096 + q * 32 + ((gg ^ ((q >> 2) & 3)) * 8);
    else
      return pr * 6144 + x * 2048 + q * 64 + ((gg ^ ((q >> 1) & 3)) * 16);
  };
  auto load_w = [&](int p0, int np) {
    const int n = np * 3 * 16 * 8;                           // (pair, gate, head, 16-byte piece)
    for (int e = tid; e < n; e += kAbThreads) {
      const int c = e & 7, hh = (e >> 3) & 15, x = (e >> 7) % 3, pr = (e >> 7) / 3;
      const int p = p0 + pr, l = p / d.NT, h = (p % d.NT) * 16 + hh;
      T v[K];
      uint4 u = make_uint4(0, 0, 0, 0);
      if (h < d.H) {
        const T* w = (const T*)(x == 0 ? a.W[0] : x == 1 ? a.W[1] : a.W[2]);
        u = *reinterpret_cast<const uint4*>(w + (int64_t)l * a.swl + (int64_t)h * a.swh + k0 + K * c);
      }
      __builtin_memcpy(v, &u, 16);
#pragma unroll
      for (int i = 0; i < K; ++i) {
        // column K c + i of the tile is MFMA tile m, row rr
        const int m = sizeof(T) == 2 ? 2 * (c >> 2) + (i >> 2) : c >> 2;
        const int rr = 4 * (c & 3) + (i & 3);
        *reinterpret_cast<T*>(&wl[w_off(pr, m * 16 + rr, x, hh >> 2) + (hh & 3) * (int)sizeof(T)]) = v[i];
      }
    }
  };
  const uint32_t row_bytes = (uint32_t)((int64_t)d.T * a.sat * (int64_t)sizeof(T));
  const uint32_t p1_bytes = (uint32_t)((int64_t)d.NP * d.NT16 * 64 * 16);
  const int64_t plane = (int64_t)d.b * d.NP * d.NT16 * 64;

  const int items = d.b * d.NT16;
  const int nchunk = (d.NP + kPairs - 1) / kPairs;
  if (nchunk == 1) {
    load_w(0, d.NP);
    __syncthreads();
  }
  // the bound is uniform over the workgroup (the chunked form has barriers inside)
  for (int it0 = blockIdx.y * 8; it0 < items; it0 += gridDim.y * 8) {
    const int it = it0 + wave;
    const bool live = it < items;
    const int itc = live ? it : items - 1;
    const int b = itc / d.NT16, tl = itc - b * d.NT16, t0 = tl * 16;
    const __amdgpu_buffer_rsrc_t rOwn = buf_rsrc((const T*)(is_b ? a.B : a.A) + (int64_t)b * a.sab, row_bytes);
    const __amdgpu_buffer_rsrc_t rOth = buf_rsrc((const T*)(is_b ? a.A : a.B) + (int64_t)b * a.sab, row_bytes);
    const unsigned char* p1b = (const unsigned char*)a.p1 + (int64_t)b * d.NP * d.NT16 * 64 * 16;
    __amdgpu_buffer_rsrc_t rP[3];
    rP[0] = buf_rsrc(p1b, p1_bytes);
    if constexpr (sizeof(T) == 2) {
      rP[1] = buf_rsrc((const unsigned char*)a.p1 + plane * 16 + (int64_t)b * d.NP * d.NT16 * 64 * 8, p1_bytes / 2);
      rP[2] = rP[1];
    } else {
      rP[1] = buf_rsrc(p1b + plane * 16, p1_bytes);
      rP[2] = buf_rsrc(p1b + plane * 32, p1_bytes);
    }
    const uint32_t sh = is_b ? 16 : 0;
    const uint32_t bits_c = a.ok[(int64_t)b * d.T + min(t0 + crow, d.T - 1)] >> sh;
    const uint32_t bits_r = a.ok[(int64_t)b * d.T + min(t0 + r, d.T - 1)] >> sh;
    const uint32_t tc = (uint32_t)min(t0 + crow, d.T - 1);
    const uint32_t rb = (uint32_t)(a.sat * (int64_t)sizeof(T));             // bytes per row
    const uint32_t kb = (uint32_t)(k0 * (int)sizeof(T));
    float own[NM * 4];
    {
      uint4 u[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) u[j] = bld16(rOwn, tc * rb + cpiece * 16 + 64 * j, kb);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint4 m = to_mfma(u[j]);
        const uint32_t w[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (sizeof(T) == 2) {
            own[8 * j + 2 * i] = __uint_as_float(w[i] << 16);
            own[8 * j + 2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
          } else {
            own[4 * j + i] = __uint_as_float(w[i]);
          }
        }
      }
    }
    float acc[NM * 4];
#pragma unroll
    for (int i = 0; i < NM * 4; ++i) acc[i] = 0.f;

    struct Frag { uint4 oth[2]; uint4 p0, p2; uint4 p1; };
    auto fetch = [&](int p, Frag& f) {
      const int l = p / d.NT;
      const int lag = 1 << l;
      const bool oc = (bits_c >> l) & 1u;
      const uint32_t src = is_b ? tc + lag : tc - lag;
      const uint32_t off = oc ? src * rb + cpiece * 16 : kOob;
#pragma unroll
      for (int j = 0; j < 2; ++j) f.oth[j] = bld16(rOth, off + 64 * j, kb);
      uint32_t idx = (uint32_t)(tl * 64 + lane);
      if (is_b) {
        const uint32_t td = (uint32_t)(t0 + r + lag);
        idx = ((bits_r >> l) & 1u) ? (td >> 4) * 64 + g * 16 + (td & 15) : kOob >> 4;
      }
      const uint32_t base = (uint32_t)p * (uint32_t)d.NT16 * 64;
      f.p0 = bld16(rP[0], idx * 16, base * 16);
      if constexpr (sizeof(T) == 2) {
        const uint32_t o8 = idx == (kOob >> 4) ? kOob : idx * 8;
        const uint2 w = bld8(rP[1], o8, base * 8);
        f.p2 = make_uint4(w.x, w.y, 0, 0);
      } else {
        f.p1 = bld16(rP[1], idx * 16, base * 16);
        f.p2 = bld16(rP[2], idx * 16, base * 16);
      }
    };
    auto compute = [&](int pr, int p, const Frag& f) {
      const int l = p / d.NT;
      // a row whose edge does not exist contributes nothing to dB (its clamp limit is 0); to dA it contributes relu(A)
      const float lim = (!is_b || ((bits_r >> l) & 1u)) ? __builtin_inff() : 0.f;
      float ov[NM * 4];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint4 m = to_mfma(f.oth[j]);
        const uint32_t w[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (sizeof(T) == 2) {
            ov[8 * j + 2 * i] = __uint_as_float(w[i] << 16);
            ov[8 * j + 2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
          } else {
            ov[4 * j + i] = __uint_as_float(w[i]);
          }
        }
      }
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        f32x4 dh = {0.f, 0.f, 0.f, 0.f};
        const int q = m * 16 + r;
        if constexpr (sizeof(T) == 2) {
          const uint4 wif = *reinterpret_cast<const uint4*>(&wl[w_off(pr, q, 0, g)]);
          const uint2 wr = *reinterpret_cast<const uint2*>(&wl[w_off(pr, q, 2, g)]);
          dh = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8i16, wif), __builtin_bit_cast(v8i16, f.p0), dh,
                                                       0, 0, 0);
          // the third gate's four heads as a half-empty fragment of the same instruction (a 16x16x16 product chained
          // onto the 16x16x32 one returned wrong sums; both take the same time)
          dh = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8i16, make_uint4(wr.x, wr.y, 0, 0)),
                                                       __builtin_bit_cast(v8i16, f.p2), dh, 0, 0, 0);
        } else {
          const uint4 pv[3] = {f.p0, f.p1, f.p2};
#pragma unroll
          for (int x = 0; x < 3; ++x) {
            const uint4 w = *reinterpret_cast<const uint4*>(&wl[w_off(pr, q, x, g)]);
            const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
            const uint32_t pp[4] = {pv[x].x, pv[x].y, pv[x].z, pv[x].w};
#pragma unroll
            for (int e = 0; e < 4; ++e)
              dh = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(ww[e]), __uint_as_float(pp[e]), dh, 0, 0, 0);
          }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float x = __builtin_amdgcn_fmed3f(own[4 * m + i] + ov[4 * m + i], 0.f, lim);
          if constexpr (sizeof(T) == 2) x = round_hi(x);
          acc[4 * m + i] = __builtin_fmaf(x, dh[i], acc[4 * m + i]);
        }
      }
    };
    for (int ch = 0; ch < nchunk; ++ch) {
      const int p0 = ch * kPairs, np = min(kPairs, d.NP - p0);
      if (nchunk > 1) {
        __syncthreads();
        load_w(p0, np);
        __syncthreads();
      }
      Frag fx, fy;
      fetch(p0, fx);
      for (int pr = 0; pr < np; pr += 2) {
        if (pr + 1 < np) fetch(p0 + pr + 1, fy);
        compute(pr, p0 + pr, fx);
        if (pr + 1 < np) {
          if (pr + 2 < np) fetch(p0 + pr + 2, fx);
          compute(pr + 1, p0 + pr + 1, fy);
        }
      }
    }
    const int t = t0 + r;
    if (live && t < d.T) {
      OT* o = (OT*)(is_b ? a.dB : a.dA) + (int64_t)b * a.sgb + (int64_t)t * a.sgt + k0;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        OT* oj = o + (4 * j + g) * K;
        float v[K];
#pragma unroll
        for (int i = 0; i < K; ++i) v[i] = 2.f * acc[K * j + i];
        if constexpr (sizeof(OT) == 2) {
          uint32_t w[K / 2];
#pragma unroll
          for (int i = 0; i < K / 2; ++i) w[i] = pack_bf16x2(v[2 * i], v[2 * i + 1]);
          __builtin_memcpy(__builtin_assume_aligned(oj, 2 * K), w, 2 * K);
        } else {
#pragma unroll
          for (int i = 0; i < K / 4; ++i)
            *reinterpret_cast<float4*>(oj + 4 * i) = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
        }
      }
    }
  }
}

// ---- dW and db ---------------------------------------------------------------------------------------------------
// One workgroup (4 waves) owns 64 columns of one (level, head group) pair over one range of position blocks; the waves
// take the range's blocks in turn. bf16: a block is 32 positions; a wave loads its A and lagged B rows coalesced, forms
// hid, writes it row-major into its own 5 KB of LDS and reads it back transposed (ds_read_tr16_b64) as the MFMA operand
// whose contraction runs over positions -- no barrier, a wave's LDS operations complete in order. fp32: a block is 16
// positions and the 16x16x4 operand is loaded directly (one element per lane). The column-tile-0 workgroups also
// multiply by ones: db.
// Bound: VALU (forming hid, ~6.5 instructions per element) and the re-read of the rows for every level.
struct WArgs {
  const void* A;
  const void* B;
  int64_t sab, sat;
  const uint4* p2;
  const uint32_t* ok;
  float* part;                  // [split][3][n_lv][H][GH], then [split][3][n_lv][H]
  int nsplit, per;              // position blocks (over all batch rows) per split
  Dims d;
};

constexpr int kWThreads = 256;
constexpr int kHidRow = 160;    // padded LDS row of 64 bf16: four rows a transposed read takes start 8 banks apart

template <typename T>
__global__ __launch_bounds__(kWThreads, 3) void gate_bwd_w(WArgs a) {
  constexpr int TB = Lay<T>::TB;
  __shared__ __align__(16) unsigned char lds[4 * 32 * kHidRow];          // also the waves' sums at the end (16 KB)
  const Dims& d = a.d;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int k0 = blockIdx.x * 64, p = blockIdx.y, l = p / d.NT, nt = p % d.NT, lag = 1 << l;
  const int q0 = blockIdx.z * a.per, q1 = min(q0 + a.per, d.b * d.NBK);
  const uint32_t row_bytes = (uint32_t)((int64_t)d.T * a.sat * (int64_t)sizeof(T));
  const uint32_t rb = (uint32_t)(a.sat * (int64_t)sizeof(T));
  const uint32_t kb = (uint32_t)(k0 * (int)sizeof(T));
  const bool bias = blockIdx.x == 0;

  f32x4 acc[4][3], accb[3];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int x = 0; x < 3; ++x) acc[c][x] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int x = 0; x < 3; ++x) accb[x] = f32x4{0.f, 0.f, 0.f, 0.f};

  if constexpr (sizeof(T) == 2) {
    unsigned char* hl = lds + wave * 32 * kHidRow;
    const int lrow = lane >> 3, lpiece = lane & 7;
    uint4 av[4], bv[4], pv[3], pn[3];
    uint32_t bits[4];
    auto row_of = [&](int q, int i, int& b) {
      b = q / d.NBK;
      return (q - b * d.NBK) * TB + 8 * i + lrow;
    };
    auto fetch_bits = [&](int q) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        int b;
        const int t = row_of(min(q, q1 - 1), i, b);
        bits[i] = a.ok[(int64_t)b * d.T + min(t, d.T - 1)];
      }
    };
    auto fetch = [&](int q) {
      const int b = q / d.NBK;
      const __amdgpu_buffer_rsrc_t rA = buf_rsrc((const T*)a.A + (int64_t)b * a.sab, row_bytes);
      const __amdgpu_buffer_rsrc_t rB = buf_rsrc((const T*)a.B + (int64_t)b * a.sab, row_bytes);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        int bb;
        const int t = row_of(q, i, bb);
        const bool in = t < d.T, ok = in && ((bits[i] >> l) & 1u);
        av[i] = bld16(rA, in ? (uint32_t)t * rb + lpiece * 16 : kOob, kb);
        bv[i] = bld16(rB, ok ? (uint32_t)(t - lag) * rb + lpiece * 16 : kOob, kb);
      }
    };
    auto fetch_p = [&](int q) {
      const int b = q / d.NBK, blk = q - b * d.NBK;
#pragma unroll
      for (int x = 0; x < 3; ++x)
        pn[x] = a.p2[((((int64_t)b * d.NP + p) * 3 + x) * d.NBK + blk) * 64 + lane];
    };
    int q = q0 + wave;
    if (q < q1) {
      fetch_bits(q);
      fetch(q);
      fetch_p(q);
      fetch_bits(q + 4);
    }
    for (; q < q1; q += 4) {
#pragma unroll
      for (int x = 0; x < 3; ++x) pv[x] = pn[x];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t aw[4] = {av[i].x, av[i].y, av[i].z, av[i].w};
        const uint32_t bw[4] = {bv[i].x, bv[i].y, bv[i].z, bv[i].w};
        uint32_t hw[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x0 = round_hi(fmaxf(__uint_as_float(aw[e] << 16) + __uint_as_float(bw[e] << 16), 0.f));
          const float x1 = round_hi(fmaxf(__uint_as_float(aw[e] & 0xffff0000u) + __uint_as_float(bw[e] & 0xffff0000u), 0.f));
          hw[e] = pack_bf16x2(x0 * x0, x1 * x1);
        }
        *reinterpret_cast<uint4*>(hl + (8 * i + lrow) * kHidRow + lpiece * 16) = make_uint4(hw[0], hw[1], hw[2], hw[3]);
      }
      if (q + 4 < q1) {                                      // uniform: the next block's rows fly during the products
        fetch(q + 4);
        fetch_p(q + 4);
        fetch_bits(q + 8);
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        // lane (r, g): positions 8 g .. 8 g + 7 of column 16 c + r; each 16-lane group reads 4 rows x 16 columns and
        // gets them transposed
        typedef __attribute__((address_space(3))) v4i16* lds4;
        const unsigned char* src = hl + (8 * g + (r >> 2)) * kHidRow + c * 32 + (r & 3) * 8;
        const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(src));
        const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(src + 4 * kHidRow));
        const v8i16 hv = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
        for (int x = 0; x < 3; ++x)
          acc[c][x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8i16, pv[x]), hv, acc[c][x], 0, 0, 0);
      }
      if (bias) {
        const v8i16 one = {0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80};
#pragma unroll
        for (int x = 0; x < 3; ++x)
          accb[x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8i16, pv[x]), one, accb[x], 0, 0, 0);
      }
    }
  } else {
    for (int q = q0 + wave; q < q1; q += 4) {
      const int b = q / d.NBK, blk = q - b * d.NBK;
      const __amdgpu_buffer_rsrc_t rA = buf_rsrc((const T*)a.A + (int64_t)b * a.sab, row_bytes);
      const __amdgpu_buffer_rsrc_t rB = buf_rsrc((const T*)a.B + (int64_t)b * a.sab, row_bytes);
      uint4 pv[3];
#pragma unroll
      for (int x = 0; x < 3; ++x) pv[x] = a.p2[((((int64_t)b * d.NP + p) * 3 + x) * d.NBK + blk) * 64 + lane];
      float hid[4][4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int t = blk * TB + 4 * g + m;
        const bool in = t < d.T;
        const bool ok = in && ((a.ok[(int64_t)b * d.T + (in ? t : d.T - 1)] >> l) & 1u);
        const uint32_t ao = in ? (uint32_t)t * rb + r * 4 : kOob, bo = ok ? (uint32_t)(t - lag) * rb + r * 4 : kOob;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float x = fmaxf(bld4f(rA, ao, kb + 64 * c) + bld4f(rB, bo, kb + 64 * c), 0.f);
          hid[m][c] = x * x;
        }
      }
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int x = 0; x < 3; ++x) {
          const float pe = __uint_as_float(m == 0 ? pv[x].x : m == 1 ? pv[x].y : m == 2 ? pv[x].z : pv[x].w);
#pragma unroll
          for (int c = 0; c < 4; ++c) acc[c][x] = __builtin_amdgcn_mfma_f32_16x16x4f32(pe, hid[m][c], acc[c][x], 0, 0, 0);
          if (bias) accb[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(pe, 1.f, accb[x], 0, 0, 0);
        }
    }
  }

  // the waves' sums added in wave order, a gate at a time (a wave's 64 columns x 16 heads: 4 KB)
  float* sum = (float*)lds;
  const int64_t nW = (int64_t)d.n_lv * d.H * d.GH, nb = (int64_t)d.n_lv * d.H;
  float* pw = a.part + (int64_t)blockIdx.z * 3 * nW;
  float* pb = a.part + (int64_t)a.nsplit * 3 * nW + (int64_t)blockIdx.z * 3 * nb;
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[wave * 1024 + (4 * g + i) * 64 + 16 * c + r] = acc[c][x][i];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int e = tid + 256 * j, h = nt * 16 + (e >> 6), k = k0 + (e & 63);
      const float v = (sum[e] + sum[1024 + e]) + (sum[2048 + e] + sum[3072 + e]);
      if (h < d.H) pw[x * nW + ((int64_t)l * d.H + h) * d.GH + k] = v;
    }
  }
  if (bias) {                                                // uniform
    __syncthreads();
    if (r == 0)
#pragma unroll
      for (int x = 0; x < 3; ++x)
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[wave * 48 + x * 16 + 4 * g + i] = accb[x][i];
    __syncthreads();
    if (tid < 48) {
      const int x = tid >> 4, h = nt * 16 + (tid & 15);
      if (h < d.H) pb[x * nb + (int64_t)l * d.H + h] = (sum[tid] + sum[48 + tid]) + (sum[96 + tid] + sum[144 + tid]);
    }
  }
}

// dW_x and db_x of `levels` levels (those from n_lv on are zeros) from the splits' sums, rounded once
template <typename OT>
__global__ __launch_bounds__(256) void gate_bwd_reduce(const float* part, int nsplit, int64_t nW, int64_t nb, int64_t fW,
                                                       int64_t fb, OT* dWi, OT* dWf, OT* dWr, OT* dbi, OT* dbf, OT* dbr) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  const int x = blockIdx.y;
  OT* W = x == 0 ? dWi : x == 1 ? dWf : dWr;
  OT* B = x == 0 ? dbi : x == 1 ? dbf : dbr;
  if (i < fW) {
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    if (i < nW) {
      const float* p = part + (int64_t)x * nW + i;
      for (int j = 0; j < nsplit; ++j) {
        const float4 v = *reinterpret_cast<const float4*>(p + (int64_t)j * 3 * nW);
        s[0] += v.x;
        s[1] += v.y;
        s[2] += v.z;
        s[3] += v.w;
      }
    }
    if constexpr (sizeof(OT) == 2)
      *reinterpret_cast<uint2*>(W + i) = make_uint2(pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3]));
    else
      *reinterpret_cast<float4*>(W + i) = make_float4(s[0], s[1], s[2], s[3]);
  }
  if (i < fb) {
    const float* p = part + (int64_t)nsplit * 3 * nW + (int64_t)x * nb;
    for (int e = 0; e < 4; ++e) {
      if (i + e >= fb) break;
      float s = 0.f;
      if (i + e < nb)
        for (int j = 0; j < nsplit; ++j) s += p[(int64_t)j * 3 * nb + i + e];
      Elem<OT>::store(B + i + e, s);
    }
  }
}

Dims dims_of(int dtype, int b, int T, int GH, int H, int n_lv) {
  const int NT = (H + 15) / 16, TB = dtype == DH_BF16 ? Lay<bf16_t>::TB : Lay<float>::TB;
  return Dims{b, T, GH, H, n_lv, NT, n_lv * NT, (T + 15) / 16, (T + TB - 1) / TB};
}

// Row ranges of gate_bwd_w: enough workgroups for ~4 per CU, each range at least 8 position blocks (two per wave).
int splits_of(const Dims& d) {
  const int64_t wgs = (int64_t)(d.GH / 64) * d.NP, blocks = (int64_t)d.b * d.NBK;
  int64_t s = (1024 + wgs - 1) / wgs;
  s = s < blocks / 8 ? s : blocks / 8;
  return (int)(s < 1 ? 1 : s);
}

struct Space {
  int64_t p1, p2, ok, part, bytes;     // byte offsets
};

Space space_of(int dtype, const Dims& d) {
  const int64_t u1 = (int64_t)d.b * d.NP * d.NT16 * 64, u2 = (int64_t)d.b * d.NP * 3 * d.NBK * 64;
  auto up = [](int64_t v) { return (v + 255) / 256 * 256; };
  Space s;
  s.p1 = 0;
  s.p2 = s.p1 + up(u1 * (dtype == DH_BF16 ? 24 : 48));
  s.ok = s.p2 + up(u2 * 16);
  s.part = s.ok + up((int64_t)d.b * d.T * 4);
  s.bytes = s.part + up((int64_t)splits_of(d) * 3 * d.n_lv * d.H * (d.GH + 1) * 4);
  return s;
}

bool aligned(const void* p, uintptr_t n) { return ((uintptr_t)p % n) == 0; }

template <typename T, typename OT>
void run_all(const PackArgs& pa, const AbArgs& aa, const WArgs& wa, int levels, void* const (&dw)[6], hipStream_t s) {
  const Dims& d = pa.d;
  const size_t lds = (size_t)3 * d.H * (kPackRows + 16 / sizeof(T)) * sizeof(T);
  gate_bwd_pack<T><<<dim3((d.T + kPackRows - 1) / kPackRows, d.n_lv, d.b), 256, lds, s>>>(pa);
  // two workgroups per CU (72 KB of LDS each), every workgroup with as many row tiles as that leaves it
  const int kt = d.GH / Lay<T>::KT, tiles = (d.b * d.NT16 + 7) / 8;
  int groups = (512 + 2 * kt - 1) / (2 * kt);
  groups = groups < tiles ? groups : tiles;
  gate_bwd_ab<T, OT><<<dim3(kt, groups, 2), kAbThreads, 0, s>>>(aa);
  gate_bwd_w<T><<<dim3(d.GH / 64, d.NP, wa.nsplit), kWThreads, 0, s>>>(wa);
  const int64_t nW = (int64_t)d.n_lv * d.H * d.GH, nb = (int64_t)d.n_lv * d.H;
  const int64_t fW = (int64_t)levels * d.H * d.GH, fb = (int64_t)levels * d.H;
  gate_bwd_reduce<OT><<<dim3((unsigned)((fW / 4 + 255) / 256), 3), 256, 0, s>>>(
      wa.part, wa.nsplit, nW, nb, fW, fb, (OT*)dw[0], (OT*)dw[1], (OT*)dw[2], (OT*)dw[3], (OT*)dw[4], (OT*)dw[5]);
}

int check_dims(const char* who, int dtype, int b, int T, int GH, int H, int n_lv) {
  DH_REQUIRE(dtype == DH_F32 || dtype == DH_BF16, DH_ERR_UNSUPPORTED_DTYPE, "%s: dtype %d", who, dtype);
  DH_REQUIRE(b >= 1 && b <= 65535 && T >= 1, DH_ERR_INVALID_ARG, "%s: b=%d (1..65535) T=%d must be >= 1", who, b, T);
  DH_REQUIRE(GH >= 64 && GH % 64 == 0, DH_ERR_UNSUPPORTED_SHAPE, "%s: GH=%d not a multiple of 64", who, GH);
  DH_REQUIRE(H >= 1 && H <= 64, DH_ERR_UNSUPPORTED_SHAPE, "%s: H=%d not in [1,64]", who, H);
  DH_REQUIRE(n_lv >= 1 && n_lv <= 16, DH_ERR_UNSUPPORTED_SHAPE, "%s: n_lv=%d not in [1,16]", who, n_lv);
  // one batch row of a dP plane stays within a buffer descriptor's range, the block count within an int
  const Dims d = dims_of(dtype, b, T, GH, H, n_lv);
  DH_REQUIRE((int64_t)d.NP * d.NT16 * 64 * 16 < ((int64_t)1 << 31) && (int64_t)b * d.NBK < ((int64_t)1 << 30) &&
                 (int64_t)b * d.NT16 < ((int64_t)1 << 30),
             DH_ERR_UNSUPPORTED_SHAPE, "%s: b=%d T=%d n_lv=%d H=%d too large", who, b, T, n_lv, H);
  return DH_OK;
}

}  // namespace

extern "C" int64_t dh_gate_preacts_bwd_workspace_bytes(int dtype, int b, int T, int GH, int H, int n_lv) {
  if (check_dims("dh_gate_preacts_bwd_workspace_bytes", dtype, b, T, GH, H, n_lv)) return -1;
  return space_of(dtype, dims_of(dtype, b, T, GH, H, n_lv)).bytes;
}

extern "C" int dh_gate_preacts_bwd_ws(int dtype, const void* A, const void* B, int64_t stride_ab, int64_t stride_at,
                                      const void* Wi, const void* Wf, const void* Wr, int64_t stride_wl,
                                      int64_t stride_wh, const void* dPi, const void* dPf, const void* dPr,
                                      int64_t stride_pb, int64_t stride_pt, int64_t stride_pl, int64_t stride_ph,
                                      const void* mask, int64_t stride_mb, int64_t stride_mt, int64_t stride_ml,
                                      int out_dtype, void* dA, void* dB, int64_t stride_gb, int64_t stride_gt, void* dWi, void* dWf, void* dWr, void* dbi,
                                      void* dbf, void* dbr, int levels, int b, int T, int GH, int H, int n_lv,
                                      void* workspace, int64_t workspace_bytes, void* stream) {
  const char* who = "dh_gate_preacts_bwd_ws";
  const int st = check_dims(who, dtype, b, T, GH, H, n_lv);
  if (st) return st;
  DH_REQUIRE(out_dtype == DH_F32 || (out_dtype == DH_BF16 && dtype == DH_BF16), DH_ERR_UNSUPPORTED_DTYPE,
             "%s: gradients of dtype %d for inputs of dtype %d", who, out_dtype, dtype);
  DH_REQUIRE(A && B && Wi && Wf && Wr && dPi && dPf && dPr && dA && dB && dWi && dWf && dWr && dbi && dbf && dbr,
             DH_ERR_INVALID_ARG, "%s: null pointer argument", who);
  DH_REQUIRE(stride_gt >= GH && stride_gb >= 0 && stride_gt % 8 == 0 && stride_gb % 8 == 0, DH_ERR_INVALID_ARG,
             "%s: gradient row stride %lld", who, (long long)stride_gt);
  DH_REQUIRE(levels >= n_lv && levels <= 64, DH_ERR_INVALID_ARG, "%s: levels=%d below n_lv=%d", who, levels, n_lv);
  const int vec = dtype == DH_BF16 ? 8 : 4;
  const int64_t esz = dtype == DH_BF16 ? 2 : 4;
  DH_REQUIRE(aligned(A, 16) && aligned(B, 16) && aligned(Wi, 16) && aligned(Wf, 16) && aligned(Wr, 16) &&
                 stride_at % vec == 0 && stride_ab % vec == 0 && stride_wl % vec == 0 && stride_wh % vec == 0 &&
                 aligned(dA, 16) && aligned(dB, 16) && aligned(dWi, 16) && aligned(dWf, 16) && aligned(dWr, 16),
             DH_ERR_INVALID_ARG, "%s: A/B/W rows and the gradients need 16-byte alignment", who);
  DH_REQUIRE(stride_at >= GH && stride_wh >= GH, DH_ERR_INVALID_ARG, "%s: strides overlap rows", who);
  DH_REQUIRE((int64_t)T * stride_at * esz < ((int64_t)1 << 31), DH_ERR_UNSUPPORTED_SHAPE,
             "%s: one batch row of A/B exceeds 2 GiB", who);
  const Dims d = dims_of(dtype, b, T, GH, H, n_lv);
  const Space sp = space_of(dtype, d);
  DH_REQUIRE(workspace && aligned(workspace, 16) && workspace_bytes >= sp.bytes, DH_ERR_INVALID_ARG,
             "%s: workspace of %lld bytes, %lld needed (16-byte aligned)", who, (long long)workspace_bytes,
             (long long)sp.bytes);
  unsigned char* ws = (unsigned char*)workspace;
  const int nsplit = splits_of(d);
  const int64_t blocks = (int64_t)d.b * d.NBK;
  const bool wide = stride_pt == 1 && aligned(dPi, 16) && aligned(dPf, 16) && aligned(dPr, 16) &&
                    stride_pb % vec == 0 && stride_pl % vec == 0 && stride_ph % vec == 0;
  PackArgs pa{{dPi, dPf, dPr}, stride_pb, stride_pt, stride_pl, stride_ph, mask, stride_mb, stride_mt, stride_ml,
              ws + sp.p1, (uint4*)(ws + sp.p2), (uint32_t*)(ws + sp.ok), wide, d};
  AbArgs aa{A, B, stride_ab, stride_at, {Wi, Wf, Wr}, stride_wl, stride_wh, ws + sp.p1, (const uint32_t*)(ws + sp.ok),
            dA, dB, stride_gb, stride_gt, d};
  WArgs wa{A, B, stride_ab, stride_at, (const uint4*)(ws + sp.p2), (const uint32_t*)(ws + sp.ok), (float*)(ws + sp.part),
           nsplit, (int)((blocks + nsplit - 1) / nsplit), d};
  void* const dw[6] = {dWi, dWf, dWr, dbi, dbf, dbr};
  hipStream_t s = (hipStream_t)stream;
  if (dtype == DH_F32) run_all<float, float>(pa, aa, wa, levels, dw, s);
  else if (out_dtype == DH_F32) run_all<bf16_t, float>(pa, aa, wa, levels, dw, s);
  else run_all<bf16_t, bf16_t>(pa, aa, wa, levels, dw, s);
  return dh_check_launch(who);
}
