// Weight gradients of bias-free linear layers, gfx950: dW_s[n,k] = sum_m dY_s[m,n] X_s[m,k], bf16 operands, fp32 sums.
//
// The contraction runs over rows, the slow dimension of both operands: an MFMA fragment wants 8 consecutive rows of one
// column in a lane. Tiles of 64 rows x 128 columns (32 x 256) are staged row-major in LDS as they come (16-byte loads, no
// transpose in registers) and the fragments are read transposed (ds_read_tr16_b64: a 16-lane group reads 4 rows x 16 columns and
// each lane receives 4 rows of its column). The four rows of such a read would share their banks at 256-byte rows, so the
// 32-byte granule q of row m is kept at q ^ (m & 3).
// A workgroup (4 waves) owns 128 x 128 outputs (64 x 64 a wave) or 128 x 256 (64 x 128 a wave) over one range of rows; up
// to four layers with the same rows go into one launch (a mixer's four projections: 256 or 128 tiles). With fewer tiles
// than workgroup slots the rows are split and a second launch adds the ranges' fp32 sums in order and rounds once; the same
// inputs give the same bits. Consecutive work items (the tiles of one layer and range, which read the same rows) go to one
// XCD.
// Bound: LDS (the fragment reads and the staging stores, see tile_k) beside the matrix cores. Measured on MI355X, four
// 1024 x 1024 gradients: called in a row on the same rows 152 us at 16384 rows (170 with the 128-wide tile), 57 at 4096, the
// library's four 453 and 124; within a training layer's pass, traced, 153-171 + 13 for the reduction at 16384 rows (over
// boxes; 745-900 TFLOP/s), 50 + 8 at 4096.
#include "dh_common.h"

namespace {

typedef short v8i16 __attribute__((ext_vector_type(8)));
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16* lds4;

constexpr int kThreads = 256, kMaxSeg = 4, kTileN = 128, kStep = 64;
constexpr uint32_t kOob = 0x80000000u;

struct Seg {
  const bf16_t* X;
  const bf16_t* dY;
  int64_t ldx, ldy;
  bf16_t* dW;
  int64_t part;                                  // first element of the layer in a range's partial sums
  int N, K, kt, tiles, first;                    // column tiles of K, tiles, first tile of the layer in the launch
};

struct WgradArgs {
  Seg seg[kMaxSeg];
  int nseg, M, nsplit, per, tiles;               // rows per range (a multiple of kStep), tiles of all layers
  float* part;                                   // [nsplit][all outputs], null when nsplit is 1
  int64_t psize;
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

// TK: 16-column MFMA tiles of a wave along K (64 x 16 TK outputs); ROWS: rows of a step
template <int TK, int ROWS>
__global__ __launch_bounds__(kThreads, 2) void wgrad_kernel(WgradArgs a) {
  constexpr int BK = 32 * TK;                      // workgroup tile: kTileN x BK
  constexpr int RY = kTileN * 2, RX = BK * 2;      // bytes of an LDS row
  constexpr int CX = BK / 8;                       // 16-byte chunks of a row of X
  constexpr int NY = ROWS / 16, NX = ROWS * CX / kThreads;
  static_assert(ROWS % 32 == 0 && kThreads % CX == 0 && ROWS * CX % kThreads == 0, "");
  __shared__ __align__(16) unsigned char ldsy[2][ROWS * RY], ldsx[2][ROWS * RX];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  // item = (layer, range, tile); each XCD (block id mod 8) takes a contiguous run of items
  const int total = a.tiles * a.nsplit, run = (total + 7) >> 3;
  const int item = (blockIdx.x & 7) * run + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= run || item >= total) return;
  Seg s = a.seg[0];
#pragma unroll
  for (int i = 1; i < kMaxSeg; ++i)
    if (i < a.nseg && item >= a.seg[i].first * a.nsplit) s = a.seg[i];
  const int local = item - s.first * a.nsplit, split = local / s.tiles, tile = local - split * s.tiles;
  const int n0 = (tile / s.kt) * kTileN, k0 = (tile % s.kt) * BK;
  const int m0 = split * a.per, m1 = min(m0 + a.per, a.M);

  // staging: thread -> 16-byte chunk cy (cx) of rows ry0 (rx0) and on; columns past N / K and rows past M read zeros
  const int cy = tid & 15, ry0 = tid >> 4, cx = tid % CX, rx0 = tid / CX;
  const uint32_t rbx = (uint32_t)(s.ldx * 2), rby = (uint32_t)(s.ldy * 2);
  const __amdgpu_buffer_rsrc_t rX = buf_rsrc(s.X, (uint32_t)((int64_t)(a.M - 1) * rbx + 2 * s.K));
  const __amdgpu_buffer_rsrc_t rY = buf_rsrc(s.dY, (uint32_t)((int64_t)(a.M - 1) * rby + 2 * s.N));
  const bool okx = k0 + 8 * cx < s.K, oky = n0 + 8 * cy < s.N;
  uint4 xv[NX], yv[NY];
  auto fetch = [&](int m) {
#pragma unroll
    for (int i = 0; i < NY; ++i) {
      const int row = m + ry0 + 16 * i;
      const uint32_t o = oky && row < m1 ? (uint32_t)row * rby + (uint32_t)(n0 + 8 * cy) * 2 : kOob;
      yv[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rY, o, 0, 0));
    }
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int row = m + rx0 + (kThreads / CX) * i;
      const uint32_t o = okx && row < m1 ? (uint32_t)row * rbx + (uint32_t)(k0 + 8 * cx) * 2 : kOob;
      xv[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rX, o, 0, 0));
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NY; ++i) {
      const int row = ry0 + 16 * i;
      *reinterpret_cast<uint4*>(&ldsy[buf][row * RY + (((cy >> 1) ^ (row & 3)) << 5) + (cy & 1) * 16]) = yv[i];
    }
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int row = rx0 + (kThreads / CX) * i;
      *reinterpret_cast<uint4*>(&ldsx[buf][row * RX + (((cx >> 1) ^ (row & 3)) << 5) + (cx & 1) * 16]) = xv[i];
    }
  };

  f32x4 acc[4][TK];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < TK; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int wn = (wave >> 1) * 64, wk = (wave & 1) * 16 * TK;
  // fragment of columns col .. col + 15, rows 32 ss + 8 g .. + 7: this lane's address within the 4-row reads
  auto frag = [&](const unsigned char* t, int rb, int ss, int col) -> v8i16 {
    const int row = 32 * ss + 8 * g + (r >> 2);
    const unsigned char* p = t + row * rb + (((col >> 4) ^ (r >> 2)) << 5) + (r & 3) * 8;
    const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(p));
    const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(p + 4 * rb));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto compute = [&](int buf) {
#pragma unroll
    for (int ss = 0; ss < ROWS / 32; ++ss) {
      v8i16 fy[4], fx[TK];
#pragma unroll
      for (int i = 0; i < 4; ++i) fy[i] = frag(ldsy[buf], RY, ss, wn + 16 * i);
#pragma unroll
      for (int j = 0; j < TK; ++j) fx[j] = frag(ldsx[buf], RX, ss, wk + 16 * j);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < TK; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fy[i], fx[j], acc[i][j], 0, 0, 0);
    }
  };

  if (m0 < m1) {                                 // uniform; an empty range adds zeros
    fetch(m0);
    store(0);
    __syncthreads();
    int buf = 0;
    for (int m = m0; m < m1; m += ROWS) {
      const bool more = m + ROWS < m1;           // uniform
      if (more) fetch(m + ROWS);
      compute(buf);
      if (more) store(buf ^ 1);
      __syncthreads();
      buf ^= 1;
    }
  }

  // C fragment: column (k) lane % 16, rows (n) 4 g + e
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < TK; ++j) {
      const int k = k0 + wk + 16 * j + r;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int n = n0 + wn + 16 * i + 4 * g + e;
        if (n >= s.N || k >= s.K) continue;
        const int64_t at = (int64_t)n * s.K + k;
        if (a.part)
          a.part[(int64_t)split * a.psize + s.part + at] = acc[i][j][e];
        else
          s.dW[at] = f32_to_bf16(acc[i][j][e]);
      }
    }
}

// the ranges' sums in order, rounded once; 4 outputs per thread (a layer's outputs are a multiple of 64)
__global__ __launch_bounds__(256) void wgrad_reduce(WgradArgs a) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= a.psize) return;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
  for (int j = 0; j < a.nsplit; ++j) {
    const float4 p = *reinterpret_cast<const float4*>(a.part + (int64_t)j * a.psize + i);
    v[0] += p.x;
    v[1] += p.y;
    v[2] += p.z;
    v[3] += p.w;
  }
  bf16_t* o = a.seg[0].dW;
  int64_t base = 0;
#pragma unroll
  for (int s = 1; s < kMaxSeg; ++s)
    if (s < a.nseg && i >= a.seg[s].part) {
      o = a.seg[s].dW;
      base = a.seg[s].part;
    }
  const uint32_t lo = (uint32_t)f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16);
  const uint32_t hi = (uint32_t)f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16);
  *reinterpret_cast<uint2*>(o + (i - base)) = make_uint2(lo, hi);
}

bool aligned(const void* p, uintptr_t n) { return ((uintptr_t)p % n) == 0; }

// Row ranges: up to the 512 workgroups the chip holds (two per CU, 64 KB of LDS each), each range at least 8 row steps.
int splits_of(int M, int tiles) {
  int s = 512 / tiles;
  const int most = M / (8 * kStep);
  if (s > most) s = most;
  return s < 1 ? 1 : s;
}

// Tile width along K: 256 columns from 6144 rows on. The wide tile reads 12 fragments per 32 MFMAs where the 128-wide one
// reads 8 per 16, but has half the tiles, so twice the row ranges and partial sums: four 1024 x 1024 gradients with the
// reduction 59 us against 57 at 4096 rows, 74 against 75 at 6144, 90 against 93 at 8192, 152 against 170 at 16384. Widths
// that a 256-column tile would pad keep the narrow one.
int tile_k(int M, int nseg, const int* K) {
  for (int s = 0; s < nseg; ++s)
    if (K[s] % 256 != 0) return 128;
  return M >= 6144 ? 256 : 128;
}

int plan(const char* who, int M, int nseg, const int* N, const int* K, int* tiles, int64_t* outputs) {
  DH_REQUIRE(M >= 1 && nseg >= 1 && nseg <= kMaxSeg && N && K, DH_ERR_INVALID_ARG, "%s: M=%d nseg=%d (1..%d)", who, M, nseg,
             kMaxSeg);
  int64_t t = 0, o = 0;
  const int bk = tile_k(M, nseg, K);
  for (int s = 0; s < nseg; ++s) {
    DH_REQUIRE(N[s] >= 8 && K[s] >= 8 && N[s] % 8 == 0 && K[s] % 8 == 0, DH_ERR_UNSUPPORTED_SHAPE,
               "%s: N=%d K=%d not multiples of 8", who, N[s], K[s]);
    t += (int64_t)((N[s] + kTileN - 1) / kTileN) * ((K[s] + bk - 1) / bk);
    o += (int64_t)N[s] * K[s];
  }
  DH_REQUIRE(t < (1 << 24), DH_ERR_UNSUPPORTED_SHAPE, "%s: too many output tiles", who);
  *tiles = (int)t;
  *outputs = o;
  return DH_OK;
}

}  // namespace

extern "C" int64_t dh_wgrad_gemm_workspace_bytes(int M, int nseg, const int* N, const int* K) {
  int tiles;
  int64_t outputs;
  if (plan("dh_wgrad_gemm_workspace_bytes", M, nseg, N, K, &tiles, &outputs)) return -1;
  const int s = splits_of(M, tiles);
  return s > 1 ? outputs * 4 * s : 0;
}

extern "C" int dh_wgrad_gemm(int dtype, int M, int nseg, const void* const* X, const int64_t* ldx, const int* K,
                             const void* const* dY, const int64_t* ldy, const int* N, void* const* dW, void* workspace,
                             int64_t workspace_bytes, void* stream) {
  const char* who = "dh_wgrad_gemm";
  DH_REQUIRE(dtype == DH_BF16, DH_ERR_UNSUPPORTED_DTYPE, "%s: dtype %d (bf16 only)", who, dtype);
  WgradArgs a{};
  const int st = plan(who, M, nseg, N, K, &a.tiles, &a.psize);
  if (st) return st;
  DH_REQUIRE(X && ldx && dY && ldy && dW, DH_ERR_INVALID_ARG, "%s: null pointer argument", who);
  const int bk = tile_k(M, nseg, K);
  a.nseg = nseg;
  a.M = M;
  int first = 0;
  int64_t part = 0;
  for (int s = 0; s < nseg; ++s) {
    DH_REQUIRE(X[s] && dY[s] && dW[s] && aligned(X[s], 16) && aligned(dY[s], 16) && aligned(dW[s], 8) && ldx[s] >= K[s] &&
                   ldy[s] >= N[s] && ldx[s] % 8 == 0 && ldy[s] % 8 == 0,
               DH_ERR_INVALID_ARG, "%s: operand %d is null, misaligned (16-byte rows) or its rows overlap", who, s);
    DH_REQUIRE((int64_t)M * ldx[s] * 2 < ((int64_t)1 << 31) && (int64_t)M * ldy[s] * 2 < ((int64_t)1 << 31),
               DH_ERR_UNSUPPORTED_SHAPE, "%s: operand %d exceeds 2 GiB", who, s);
    const int kt = (K[s] + bk - 1) / bk, tiles = ((N[s] + kTileN - 1) / kTileN) * kt;
    a.seg[s] = Seg{(const bf16_t*)X[s], (const bf16_t*)dY[s], ldx[s], ldy[s], (bf16_t*)dW[s], part, N[s], K[s], kt, tiles,
                   first};
    first += tiles;
    part += (int64_t)N[s] * K[s];
  }
  a.nsplit = splits_of(M, a.tiles);
  a.per = ((M + a.nsplit - 1) / a.nsplit + kStep - 1) / kStep * kStep;
  if (a.nsplit > 1) {
    DH_REQUIRE(workspace && aligned(workspace, 16) && workspace_bytes >= a.psize * 4 * a.nsplit, DH_ERR_INVALID_ARG,
               "%s: workspace of %lld bytes, %lld needed (16-byte aligned)", who, (long long)workspace_bytes,
               (long long)(a.psize * 4 * a.nsplit));
    a.part = (float*)workspace;
  }
  hipStream_t s = (hipStream_t)stream;
  const int total = a.tiles * a.nsplit;
  const dim3 grid((unsigned)((total + 7) / 8 * 8));
  if (bk == 256)
    wgrad_kernel<8, 32><<<grid, kThreads, 0, s>>>(a);
  else
    wgrad_kernel<4, 64><<<grid, kThreads, 0, s>>>(a);
  if (a.part) wgrad_reduce<<<dim3((unsigned)((a.psize / 4 + 255) / 256)), 256, 0, s>>>(a);
  return dh_check_launch(who);
}
