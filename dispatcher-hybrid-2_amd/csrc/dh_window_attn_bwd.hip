// Gradient of the banded causal attention with interleaved rope, gfx950 (bf16, head width 64).
//
// Semantics: the autograd of reference dispatcher_hybrid/modeling_dispatcher.py:163-182 (rope, scores / sqrt(hd), banded
// softmax, value average) for the outputs dh_window_attention_train_fwd wrote. With P = softmax (recomputed from the saved
// log2-sum-exp), all sums fp32 and P, dS rounded to bf16 as matrix operands (the dtype the eager path has them in):
//   delta[t] = sum_c dO[t,c] O[t,c]
//   dV[s] = sum_t P[t,s] dO[t]      dS[t,s] = P[t,s] (dO[t] . V[s] - delta[t])
//   dQ'[t] = sum_s dS[t,s] K'[s] / sqrt(hd)      dK'[s] = sum_t dS[t,s] Q'[t] / sqrt(hd)      (primes: rotated)
// and dQ, dK rotated back. Two launches: a pre-pass (rotated queries head-major, delta), then one kernel in two forms.
//
// Work decomposition: a workgroup of 4 waves owns 64 rows of one (batch row, head) -- queries for dQ, keys for dK and dV --
// and walks the 64-row blocks of the other side inside the band; wave w owns rows 16 w .. + 15, their two operand fragments
// in registers. Both streamed blocks (keys and values, or rotated queries and dO) sit row-major in double-buffered LDS
// (rows padded to 144 bytes). Scores and dO.V come out of MFMA as C fragments with one owned row per lane column, which is
// the B-operand layout of the two products that contract over the streamed rows; their A operands, the streamed blocks
// transposed, are read with ds_read_tr16_b64 from the same LDS tiles. So nothing is transposed in registers and no value
// crosses a wave.
// Bound: VALU (~9 instructions per score and form) beside 3 (dQ) and 4 (dK, dV) MFMA products. Measured on MI355X at B 2,
// T 2048, window 1024, 16 heads: 90 us and the pre-pass 9 (58 GFLOP with the forward's), where the blockwise torch
// attention took ~390 launches and 4 ms for the two directions.
#include "dh_attn_common.h"

namespace {

constexpr int HD = 64, kB = 64, kThreads = 256, kRow = HD * 2 + 16, kKS = HD / 32, kNT = HD / 16;
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef short v8i16 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) v4i16* lds4;

struct BwdArgs {
  const bf16_t* q;              // projection rows before rope: b sb + t st + h HD
  int64_t sb, st;
  const bf16_t* kr;             // (B, H, T, HD): rotated keys, values, rotated queries (written by the pre-pass)
  const bf16_t* vr;
  bf16_t* qr;
  const bf16_t* o;              // attention output and its gradient: b ob + t ot + h HD
  const bf16_t* dO;
  int64_t ob, ot, gb, gt;
  const float* lse;             // (B, H, T)
  float* delta;                 // (B, H, T)
  const bf16_t* cos;            // (>= T, HD / 2)
  const bf16_t* sin;
  bf16_t* dq;                   // gradients: b db + t dt + h HD
  bf16_t* dk;
  bf16_t* dv;
  int64_t db, dt;
  int B, T, H, window, nblk, nwork;
  float scale, scale2;          // 1 / sqrt(hd), the same times log2 e
};

// rotated queries and delta: one thread per 16-byte chunk of a (b, t, h) row, 8 consecutive lanes a row
__global__ __launch_bounds__(kThreads) void attn_bwd_prep(BwdArgs a) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x, n = (int64_t)a.B * a.T * a.H * 8;
  const int64_t ic = i < n ? i : n - 1;
  const int c = (int)(ic & 7);
  const int64_t row = ic >> 3;
  const int h = (int)(row % a.H);
  const int64_t bt = row / a.H;
  const int t = (int)(bt % a.T), b = (int)(bt / a.T);
  const int col = h * HD + 8 * c;
  const uint4 o = ld16(a.o + (int64_t)b * a.ob + (int64_t)t * a.ot + col);
  const uint4 g = ld16(a.dO + (int64_t)b * a.gb + (int64_t)t * a.gt + col);
  const uint4 qv = rope8(ld16(a.q + (int64_t)b * a.sb + (int64_t)t * a.st + col), ld8(a.cos + (int64_t)t * (HD / 2) + 4 * c),
                         ld8(a.sin + (int64_t)t * (HD / 2) + 4 * c));
  const uint32_t ow[4] = {o.x, o.y, o.z, o.w}, gw[4] = {g.x, g.y, g.z, g.w};
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    s = __builtin_fmaf(lo_f(ow[e]), lo_f(gw[e]), s);
    s = __builtin_fmaf(hi_f(ow[e]), hi_f(gw[e]), s);
  }
  s += dpp_move<0xb1, 0xf>(s);     // lanes 1, 2 and (mirrored) 4 apart
  s += dpp_move<0x4e, 0xf>(s);
  s += dpp_move<0x141, 0xf>(s);
  if (i >= n) return;
  const int64_t hm = ((int64_t)b * a.H + h) * a.T + t;
  *reinterpret_cast<uint4*>(a.qr + hm * HD + 8 * c) = qv;
  if (c == 0) a.delta[hm] = s;
}

struct BwdLds {
  __align__(16) unsigned char tile[2][2][kB * kRow];                     // [buffer][keys | queries, values | dO]
  __align__(16) float stat[2][2][kB];                                    // KV: log2-sum-exp and delta of the block's queries
};

// KV: dK and dV of 64 keys, else dQ of 64 queries; item w = block of 64 rows of one (batch row, head)
template <bool KV>
__device__ __forceinline__ void attn_bwd_rows(const BwdArgs& a, BwdLds& lds, int w) {
  auto& tile = lds.tile;
  auto& stat = lds.stat;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int blk = w % a.nblk, bh = w / a.nblk, h = bh % a.H, b = bh / a.H;
  const int own0 = blk * kB;
  const int town = own0 + wave * 16 + r;                                 // this lane's row
  const int tc = min(town, a.T - 1);
  const int64_t head = (int64_t)bh * a.T;
  const bf16_t* dOp = a.dO + (int64_t)b * a.gb + (int64_t)h * HD;

  // owned operands: lane (row r, k-group g) holds columns 32 s + 8 g .. + 8 of keys | queries and of values | dO
  bf16x8 f1[kKS], f2[kKS];
#pragma unroll
  for (int s = 0; s < kKS; ++s) {
    const int col = 32 * s + 8 * g;
    f1[s] = as_bf16x8(ld16((KV ? a.kr : a.qr) + (head + tc) * HD + col));
    f2[s] = as_bf16x8(ld16(KV ? a.vr + (head + tc) * HD + col : dOp + (int64_t)tc * a.gt + col));
  }
  const float lse_own = KV ? 0.f : a.lse[head + tc], delta_own = KV ? 0.f : a.delta[head + tc];

  // blocks of the other side inside the band
  int j0, j1;
  if (KV) {
    j0 = blk;
    j1 = (a.window > 0 ? min((int64_t)own0 + kB - 1 + a.window - 1, (int64_t)a.T - 1) : (int64_t)a.T - 1) / kB;
  } else {
    j0 = a.window > 0 ? max(0, own0 - a.window + 1) / kB : 0;
    j1 = min(own0 + kB - 1, a.T - 1) / kB;
  }
  uint4 x1[2], x2[2];
  float st = 0.f;
  auto fetch = [&](int j) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int idx = tid + i * kThreads, c = idx & 7, t = min(j * kB + (idx >> 3), a.T - 1);
      x1[i] = ld16((KV ? a.qr : a.kr) + (head + t) * HD + 8 * c);
      x2[i] = ld16(KV ? dOp + (int64_t)t * a.gt + 8 * c : a.vr + (head + t) * HD + 8 * c);
    }
    if (KV && tid < 2 * kB) st = (tid < kB ? a.lse : a.delta)[head + min(j * kB + (tid & (kB - 1)), a.T - 1)];
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int idx = tid + i * kThreads, off = (idx >> 3) * kRow + (idx & 7) * 16;
      *reinterpret_cast<uint4*>(&tile[buf][0][off]) = x1[i];
      *reinterpret_cast<uint4*>(&tile[buf][1][off]) = x2[i];
    }
    if (KV && tid < 2 * kB) stat[buf][tid >> 6][tid & (kB - 1)] = st;
  };
  // C fragment (streamed row 16 tau + 4 g + i, owned row r) of a streamed tile times an owned operand
  auto product = [&](const unsigned char* t, const bf16x8 (&f)[kKS], f32x4 (&out)[4]) {
#pragma unroll
    for (int tau = 0; tau < 4; ++tau) {
      out[tau] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < kKS; ++s)
        out[tau] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            *reinterpret_cast<const bf16x8*>(t + (tau * 16 + r) * kRow + (32 * s + 8 * g) * 2), f[s], out[tau], 0, 0, 0);
    }
  };
  // acc (column 16 nt + 4 g + i, owned row r) += tile^T times the bf16 pairs of p, streamed rows in the order the C fragments
  // hold them: rows 32 kk + 4 g .. + 3, then 32 kk + 16 + 4 g .. + 3
  auto accumulate = [&](const unsigned char* t, const uint32_t (&p)[8], f32x4 (&acc)[kNT]) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const bf16x8 pf = as_bf16x8(make_uint4(p[4 * kk], p[4 * kk + 1], p[4 * kk + 2], p[4 * kk + 3]));
#pragma unroll
      for (int nt = 0; nt < kNT; ++nt) {
        const unsigned char* src = t + (32 * kk + 4 * g + (r >> 2)) * kRow + nt * 32 + (r & 3) * 8;
        const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(src));
        const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(src + 16 * kRow));
        const v8i16 tv = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, tv), pf, acc[nt], 0, 0, 0);
      }
    }
  };

  f32x4 acc[kNT], accv[kNT];
#pragma unroll
  for (int nt = 0; nt < kNT; ++nt) acc[nt] = accv[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  fetch(j0);
  store(0);
  __syncthreads();
  for (int j = j0; j <= j1; ++j) {
    const int buf = (j - j0) & 1;
    const bool more = j < j1;                                            // uniform
    if (more) fetch(j + 1);
    f32x4 s4[4], d4[4];
    product(tile[buf][0], f1, s4);
    product(tile[buf][1], f2, d4);
    // a block wholly inside the band and the sequence needs no mask
    const int qlast = (KV ? j : blk) * kB + kB - 1, kfirst = (KV ? blk : j) * kB;
    const bool interior = j != blk && qlast < a.T && (a.window == 0 || qlast - kfirst < a.window);
    uint32_t p[8], ds[8];
#pragma unroll
    for (int tau = 0; tau < 4; ++tau) {
      float ls[4], dl[4];
      if constexpr (KV) {
        const float4 l4 = *reinterpret_cast<const float4*>(&stat[buf][0][tau * 16 + 4 * g]);
        const float4 e4 = *reinterpret_cast<const float4*>(&stat[buf][1][tau * 16 + 4 * g]);
        ls[0] = l4.x; ls[1] = l4.y; ls[2] = l4.z; ls[3] = l4.w;
        dl[0] = e4.x; dl[1] = e4.y; dl[2] = e4.z; dl[3] = e4.w;
      }
      float pv[4], dv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float l = KV ? ls[i] : lse_own, dd = KV ? dl[i] : delta_own;
        float pr = __builtin_amdgcn_exp2f(__builtin_fmaf(s4[tau][i], a.scale2, -l));
        if (!interior) {                                                 // uniform
          const int other = j * kB + tau * 16 + 4 * g + i;
          const int tq = KV ? other : town, tk = KV ? town : other;
          const bool ok = tk <= tq && tq < a.T && (a.window == 0 || tq - tk < a.window);
          pr = ok ? pr : 0.f;
        }
        pv[i] = pr;
        dv[i] = pr * (d4[tau][i] - dd);
      }
      p[2 * tau] = pack2(pv[0], pv[1]);
      p[2 * tau + 1] = pack2(pv[2], pv[3]);
      ds[2 * tau] = pack2(dv[0], dv[1]);
      ds[2 * tau + 1] = pack2(dv[2], dv[3]);
    }
    if constexpr (KV) accumulate(tile[buf][1], p, accv);                 // dV^T += dO^T P
    accumulate(tile[buf][0], ds, acc);                                   // dK^T += Q'^T dS, dQ^T += K'^T dS^T
    if (more) store(buf ^ 1);
    __syncthreads();
  }

  if (town < a.T) {
    const int64_t row = (int64_t)b * a.db + (int64_t)town * a.dt + (int64_t)h * HD;
    bf16_t* d1 = (KV ? a.dk : a.dq) + row;
#pragma unroll
    for (int nt = 0; nt < kNT; ++nt) {
      const int col = nt * 16 + 4 * g;
      const uint32_t cw = *reinterpret_cast<const uint32_t*>(a.cos + (int64_t)town * (HD / 2) + col / 2);
      const uint32_t sw = *reinterpret_cast<const uint32_t*>(a.sin + (int64_t)town * (HD / 2) + col / 2);
      uint32_t out[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {                                      // the rotation's transpose on each pair
        const float c = e ? hi_f(cw) : lo_f(cw), s = e ? hi_f(sw) : lo_f(sw);
        const float g0 = acc[nt][2 * e] * a.scale, g1 = acc[nt][2 * e + 1] * a.scale;
        out[e] = pack2(__builtin_fmaf(g0, c, g1 * s), __builtin_fmaf(g1, c, -(g0 * s)));
      }
      *reinterpret_cast<uint2*>(d1 + col) = make_uint2(out[0], out[1]);
      if constexpr (KV)
        *reinterpret_cast<uint2*>(a.dv + row + col) =
            make_uint2(pack2(accv[nt][0], accv[nt][1]), pack2(accv[nt][2], accv[nt][3]));
    }
  }
}

// Both forms in one launch, the key blocks (more products each) first: two launches end in a round of their own each, and a
// short sequence fills the CUs with neither (B 2, T 2048, window 1024, 16 heads: 59 + 41 us -> 90).
__global__ __launch_bounds__(kThreads, 3) void attn_bwd_kernel(BwdArgs a) {
  __shared__ BwdLds lds;
  const int per = (a.nwork + 7) >> 3;                                    // consecutive items (blocks of one head) on one XCD
  const int i = blockIdx.x >> 3;
  const bool kv = i < per;
  const int w = (blockIdx.x & 7) * per + (kv ? i : i - per);
  if (w >= a.nwork) return;
  if (kv)
    attn_bwd_rows<true>(a, lds, w);
  else
    attn_bwd_rows<false>(a, lds, w);
}

bool aligned(const void* p, uintptr_t n) { return ((uintptr_t)p % n) == 0; }

}  // namespace

extern "C" int dh_window_attention_bwd(int dtype, const void* q, int64_t stride_b, int64_t stride_t, const void* K_rot,
                                       const void* V_rows, const void* y, int64_t y_stride_b, int64_t y_stride_t,
                                       const void* dy, int64_t dy_stride_b, int64_t dy_stride_t, const float* lse,
                                       const void* rope_cos, const void* rope_sin, void* Q_rot, float* delta, void* dq,
                                       void* dk, void* dv, int64_t d_stride_b, int64_t d_stride_t, int B, int T, int H,
                                       int hd, int window, void* stream) {
  const char* who = "dh_window_attention_bwd";
  DH_REQUIRE(dtype == DH_BF16, DH_ERR_UNSUPPORTED_DTYPE, "%s: dtype %d (bf16 only)", who, dtype);
  DH_REQUIRE(hd == HD, DH_ERR_UNSUPPORTED_SHAPE, "%s: hd=%d (64)", who, hd);
  DH_REQUIRE(B >= 1 && T >= 1 && H >= 1 && window >= 0, DH_ERR_INVALID_ARG, "%s: B=%d T=%d H=%d window=%d", who, B, T, H,
             window);
  DH_REQUIRE(q && K_rot && V_rows && y && dy && lse && rope_cos && rope_sin && Q_rot && delta && dq && dk && dv,
             DH_ERR_INVALID_ARG, "%s: null pointer argument", who);
  const int64_t strides[] = {stride_b, stride_t, y_stride_b, y_stride_t, dy_stride_b, dy_stride_t, d_stride_b, d_stride_t};
  bool ok = aligned(q, 16) && aligned(K_rot, 16) && aligned(V_rows, 16) && aligned(y, 16) && aligned(dy, 16) &&
            aligned(Q_rot, 16) && aligned(dq, 8) && aligned(dk, 8) && aligned(dv, 8) && aligned(rope_cos, 8) &&
            aligned(rope_sin, 8);
  for (int64_t s : strides) ok = ok && s >= 0 && s % 8 == 0;
  for (int64_t s : {stride_t, y_stride_t, dy_stride_t, d_stride_t}) ok = ok && s >= (int64_t)H * hd;
  DH_REQUIRE(ok, DH_ERR_INVALID_ARG, "%s: rows need 16-byte alignment and strides of at least H * hd", who);
  const int nblk = (T + kB - 1) / kB;
  const int64_t nwork = (int64_t)nblk * H * B, chunks = (int64_t)B * T * H * 8;
  DH_REQUIRE(nwork < (1 << 30) && chunks < ((int64_t)1 << 38), DH_ERR_UNSUPPORTED_SHAPE, "%s: too many row blocks", who);
  const float scale = (float)(1.0 / sqrt((double)hd));
  BwdArgs a{(const bf16_t*)q, stride_b, stride_t, (const bf16_t*)K_rot, (const bf16_t*)V_rows, (bf16_t*)Q_rot,
            (const bf16_t*)y, (const bf16_t*)dy, y_stride_b, y_stride_t, dy_stride_b, dy_stride_t, lse, delta,
            (const bf16_t*)rope_cos, (const bf16_t*)rope_sin, (bf16_t*)dq, (bf16_t*)dk, (bf16_t*)dv, d_stride_b, d_stride_t,
            B, T, H, window, nblk, (int)nwork, scale, scale * 1.44269504088896341f};
  hipStream_t s = (hipStream_t)stream;
  const unsigned grid = (unsigned)((nwork + 7) / 8 * 8);
  attn_bwd_prep<<<dim3((unsigned)((chunks + kThreads - 1) / kThreads)), kThreads, 0, s>>>(a);
  attn_bwd_kernel<<<dim3(2 * grid), kThreads, 0, s>>>(a);
  return dh_check_launch(who);
}
