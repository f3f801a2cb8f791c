// One mixer layer's inference forward as one call: four launches issued from native code. A short prompt's launches take
// ~45 us of GPU time at d = 1024; issued one by one through the host bindings they took ~100 us.
#include "dh_common.h"

namespace {

int64_t up(int64_t v) { return (v + 255) / 256 * 256; }

// scratch: the projections V0, A, B, then the scanned state (b, T, d), then the gates (3, b, H, n_lv, Tp), Tp = T rounded
// up to 8 (rows start aligned whatever T is, so the gates are stored four positions at a time)
struct Space {
  int64_t proj, gates, bytes, Tp;
};

Space space_of(int dtype, int b, int T, int d, int H, int n_lv) {
  const int64_t esz = dtype == DH_BF16 ? 2 : 4;
  Space s;
  s.Tp = (T + 7) / 8 * 8;
  s.proj = up((int64_t)b * T * d * esz);
  s.gates = up((int64_t)b * H * n_lv * s.Tp * esz);
  s.bytes = 4 * s.proj + 3 * s.gates;
  return s;
}

int check_layer(const char* who, int dtype, int b, int T, int d, int H, int n_lv) {
  DH_REQUIRE(dtype == DH_F32 || dtype == DH_BF16, DH_ERR_UNSUPPORTED_DTYPE, "%s: dtype %d", who, dtype);
  DH_REQUIRE(b >= 1 && T >= 1 && (int64_t)b * T < ((int64_t)1 << 31), DH_ERR_INVALID_ARG, "%s: b=%d T=%d", who, b, T);
  DH_REQUIRE(H >= 1 && H <= 64 && d >= 64 && d % 64 == 0 && d % H == 0 && n_lv >= 1 && n_lv <= 16,
             DH_ERR_UNSUPPORTED_SHAPE, "%s: d=%d H=%d n_lv=%d", who, d, H, n_lv);
  return DH_OK;
}

}  // namespace

extern "C" int64_t dh_mixer_fwd_scratch_bytes(int dtype, int b, int T, int d, int H, int n_lv) {
  if (check_layer("dh_mixer_fwd_scratch_bytes", dtype, b, T, d, H, n_lv)) return -1;
  return space_of(dtype, b, T, d, H, n_lv).bytes;
}

extern "C" int dh_mixer_fwd(int dtype, const void* x, int64_t ldx, const void* W_in, const void* W_x, const void* W_s,
                            const void* Wi, const void* Wf, const void* Wr, const void* bi, const void* bf,
                            const void* br, const void* W_out, const void* mask, int64_t stride_mb, int64_t stride_mt,
                            int64_t stride_ml, void* y, void* scratch, int64_t scratch_bytes, int b, int T, int d, int H,
                            int n_lv, void* stream) {
  const char* who = "dh_mixer_fwd";
  int st = check_layer(who, dtype, b, T, d, H, n_lv);
  if (st) return st;
  const Space sp = space_of(dtype, b, T, d, H, n_lv);
  DH_REQUIRE(scratch && (uintptr_t)scratch % 256 == 0 && scratch_bytes >= sp.bytes, DH_ERR_INVALID_ARG,
             "%s: scratch of %lld bytes, %lld needed (256-byte aligned)", who, (long long)scratch_bytes,
             (long long)sp.bytes);
  unsigned char* base = (unsigned char*)scratch;
  void* V0 = base;
  void* A = base + sp.proj;
  void* B = base + 2 * sp.proj;
  void* V = base + 3 * sp.proj;
  void* g[3];
  for (int i = 0; i < 3; ++i) g[i] = base + 4 * sp.proj + i * sp.gates;
  const int rows = b * T;
  const void* const W[3] = {W_in, W_x, W_s};
  void* const out[3] = {V0, A, B};
  const int N[3] = {d, d, d};
  const int64_t ld[3] = {d, d, d};
  st = dh_proj_gemm(dtype, x, ldx, rows, d, 3, W, N, out, ld, stream);
  if (st) return st;
  const int64_t hd = (int64_t)H * d, gb = (int64_t)H * n_lv * sp.Tp;
  st = dh_gate_preacts_fwd(dtype, A, B, (int64_t)T * d, d, Wi, Wf, Wr, hd, d, bi, bf, br, mask, stride_mb, stride_mt,
                           stride_ml, g[0], g[1], g[2], gb, 1, sp.Tp, (int64_t)n_lv * sp.Tp, 1 | 2, b, T, d, H, n_lv,
                           stream);
  if (st) return st;
  st = dh_level_scan_fwd(dtype, g[0], g[1], g[2], gb, 1, sp.Tp, (int64_t)n_lv * sp.Tp, nullptr, 0, 0, 0, V0,
                         (int64_t)T * d, d, V, b, T, H, d / H, n_lv, 1, nullptr, 0, stream);
  if (st) return st;
  const void* const Wo[1] = {W_out};
  void* const yo[1] = {y};
  return dh_proj_gemm(dtype, V, d, rows, d, 1, Wo, N, yo, ld, stream);
}
