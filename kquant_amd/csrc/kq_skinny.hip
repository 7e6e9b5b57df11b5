// Launches of the few-row linear (kq_skinny.h): which instantiation a shape
// takes.
#include "kq_skinny.h"
#include "kq_internal.h"

namespace kq {
namespace skinny {

template <int FMT, int AT, int OUT, int MB, int R, int P, bool HALF>
static hipError_t launch(const SkinnyArgs& s, hipStream_t st) {
  const int nwin = (s.k + WIN - 1) / WIN;
  const int waves = nwin < 8 ? nwin : 8;
  const size_t lds = (size_t)waves * MB * R * 1024;
  auto kern = mx_skinny_kernel<FMT, AT, OUT, MB, R, P, HALF>;
  if (lds > 65536) {
    const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  const int64_t mtiles = (s.m + 16 * MB - 1) / (16 * MB), ntiles = ((int64_t)s.n + 16 * R - 1) / (16 * R);
  kern<<<(unsigned)(mtiles * ((ntiles + 7) / 8 * 8)), waves * 64, lds, st>>>(
      s.a, s.a_scale, s.lda, s.wq, s.ws, s.c, s.ldc, s.m, s.n, s.k, (int)mtiles);
  return hipGetLastError();
}

// Row blocks per workgroup.  One block of 16 weight rows (R = 1) puts the
// most workgroups on the chip, which is what a decode row needs (N = 12288,
// K = 7168 E4M3, one row, cold: 24 us; R = 2 / 4: 27 / 30); with 17 rows and
// more the activations outweigh the weights unless four blocks share a read
// of them (32 rows: 42.6 us against 52; 64 rows: 57 against 95), which pays
// while N / 64 workgroups still cover half the CUs.  Half windows keep R = 1
// past 16 rows: fp32 rows, N = 12288, K = 2112, 17 / 32 rows 44 / 58 us with E4M3 weights
// (171 / 172 in whole tiles), 53 at 17 with E2M1 (16 registers spill; 160), and
// the tiles' split, 46, at 32.
template <int FMT, int AT, int OUT, bool HALF>
static hipError_t launch_rows(const SkinnyArgs& s, hipStream_t st) {
  const bool wide = s.n >= 64 * 128;
  if (s.m <= 16) return launch<FMT, AT, OUT, 1, 1, 2, HALF>(s, st);
  if constexpr (AT == A_F32) {
    if (wide && !HALF) return launch<FMT, AT, OUT, 2, 4, 2, false>(s, st);
    return launch<FMT, AT, OUT, 2, 1, 2, HALF>(s, st);
  } else {
    if (s.m <= 32) {
      if (wide && !HALF) return launch<FMT, AT, OUT, 2, 4, 2, false>(s, st);
      return launch<FMT, AT, OUT, 2, 1, 2, HALF>(s, st);
    }
    if constexpr (AT == A_BF16)  // (expanding MXFP8 rows too takes more registers than there are)
      if (wide && !HALF) return launch<FMT, AT, OUT, 4, 4, 2, false>(s, st);
    return launch<FMT, AT, OUT, 4, 1, 2, HALF>(s, st);
  }
}

template <int FMT, int AT, int OUT>
static hipError_t launch_k(const SkinnyArgs& s, hipStream_t st) {
  return s.k % WIN ? launch_rows<FMT, AT, OUT, true>(s, st) : launch_rows<FMT, AT, OUT, false>(s, st);
}

}  // namespace skinny

hipError_t mx_skinny_bf16(int fmt, bool out_f32, const SkinnyArgs& s, hipStream_t st) {
  using namespace skinny;
  if (fmt == KQ_FMT_MXFP8_E4M3) return out_f32 ? launch_k<0, A_BF16, 2>(s, st) : launch_k<0, A_BF16, 0>(s, st);
  return out_f32 ? launch_k<1, A_BF16, 2>(s, st) : launch_k<1, A_BF16, 0>(s, st);
}

hipError_t mx_skinny_f32(int fmt, const SkinnyArgs& s, hipStream_t st) {
  using namespace skinny;
  return fmt == KQ_FMT_MXFP8_E4M3 ? launch_k<0, A_F32, 2>(s, st) : launch_k<1, A_F32, 2>(s, st);
}

hipError_t mx_skinny_mx(bool out_f32, const SkinnyArgs& s, hipStream_t st) {
  using namespace skinny;
  return out_f32 ? launch_rows<0, A_MXFP8, 2, false>(s, st) : launch_rows<0, A_MXFP8, 0, false>(s, st);
}

}  // namespace kq
