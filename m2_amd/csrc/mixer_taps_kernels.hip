// The mixer core on filter taps: the kernels of mixer_pair.h (L = 1024 .. 4096) and mixer_long.h (8192, 16384) that transform the
// filters of a row's channel themselves, and their C entry point.  bf16 rows.
//
// A filter's spectrum is made for all rows of its channel, and with one row to a channel it is written and read for that row alone: 32 d L
// bytes per layer beside the 16 d L of the taps, which the transform reads either way.  Here the taps go from memory into the
// first pass's layout, are transformed by the row's own threads and stay in registers as the spectrum (64 of 256, in which the next taps are
// requested as soon as the product has freed them).  It is the spectrum that the other kernels store, value by value and with its factor 1 / L,
// so that a forward has the same bits on either route (the factor's 64 multiplications a thread: L = 8192, B = 1 70.7 / 72.5 us, 4096 35.5 / 35.6,
// a forward of 12 x 768 at 4096 1629 / 1635).  What bounds it stays the vector ALU: half as many instructions again as the core
// on spectra, which the memory traffic that is gone pays for as long as no second row would share the spectrum.
//
// us, d = 768, bf16, core and its spectra (of one mixer / a twelfth of twelve mixers' at once) against the core on taps: L = 1024, B = 1
// 10.4 + 8.4 / 6 against 13.5, 2048 15.6 + 11.0 / 9 against 22.1, 4096 25.2 + 20.1 / 17.4 against 37.1, 8192 46.4 + 37.9 / 36.5 against 73.9,
// 16384 104.8 + 90.5 against 154.8; B = 2 12.5, 23.4, 41.7, 81.7, 195.4 against 16.6, 32.3, 57.6, 112.2, 289.0 (up to 5 % of both, or a loss),
// B = 3 19.0, 32.3, 56.5, 136.9, 288.6 against 25.5, 46.2, 79.7, 173.7, 421.1.  So: one row to a channel, and two where whole forwards
// gain by it too: 12 x 768, B = 2, L = 1024 1090 / 1102, 2048 1531 / 1550, 4096 2295 / 2264, 8192 4837 / 4704.  Whole forwards of 12 x 768, B = 1:
// L = 1024 1011 / 971, 2048 1230 / 1208, 4096 1793 / 1723, 8192 2814 / 2680, 16384 6030 / 5720; 24 x 1536, 2048 4786 / 4541.
// The width changes little, as both routes grow with it.  Six layers, spectra / taps: B = 1, L = 1024, 4096, 16384 960 553 / 500, 1111 / 1048,
// 3685 / 3499, 1536 804 / 770, 1834 / 1716, 6626 / 6168, 1792 918 / 878, 2230 / 2099, 8084 / 7548; B = 2, L = 4096, 8192 768 1091 / 1079, 2053 / 2011,
// 960 1629 / 1610, 3000 / 2956, 1536 2773 / 2726, 5588 / 5490, 1792 3512 / 3457, 6869 / 6786.
// fp32 rows, whose inputs take twice the registers, spill beside a spectrum (52 bytes a lane and more) and read spectra; at L = 32768 a
// half transform's inputs would have to be formed twice from all the taps.
#include "mixer_long.h"
#include "mixer_pair.h"

namespace m2 {

static int launch_mixer_taps(const void* xproj, long ldx, const float* u, const float* sw, const float* sb, const float* pbias,
                             const FilterTaps& filters, void* y, int B, int L, int d, hipStream_t s) {
  switch (L) {
#define X(LEN) case LEN: return launch_mixer_pair<Twist##LEN, uint16_t, true>(xproj, ldx, u, sw, sb, pbias, nullptr, filters, y, B, d, s);
    X(1024) X(2048) X(4096)
#undef X
#define X(LEN) case LEN: return launch_mixer_long<Twist##LEN, uint16_t, true>(xproj, ldx, u, sw, sb, pbias, nullptr, filters, y, B, d, s);
    X(8192) X(16384)
#undef X
  }
  return set_error(M2_ERR_UNSUPPORTED, "m2_mixer_core_taps_fwd: L=%d unsupported (need L a power of two in [1024, 16384])", L);
}

}  // namespace m2

using namespace m2;

extern "C" int m2_mixer_core_taps_pays(int B, int L) {
  return m2_fftconv_supported_seqlen(L) && L >= 1024 && ((B == 1 && L <= 16384) || (B == 2 && L >= 4096 && L <= 8192));
}

extern "C" int m2_mixer_core_taps_fwd(const void* xproj, long xproj_row, const float* proj_bias, const float* u, const float* short_w,
                                      const float* short_b, const float* taps, const float* const* skip_dev, int nfilters, void* y,
                                      int B, int L, int d, void* stream) {
  const char* who = "m2_mixer_core_taps_fwd";
  if (!xproj || !short_w || !short_b || !taps || !y) return set_error(M2_ERR_ARG, "%s: null pointer", who);
  if (nfilters < 1 || nfilters > 2 || (u && nfilters != 2))
    return set_error(M2_ERR_ARG, "%s: %d filters, need 1, or 2 with a second input", who, nfilters);
  if (B <= 0 || d <= 0 || d % 8 != 0) return set_error(M2_ERR_ARG, "%s: need B > 0 and d a positive multiple of 8 (B=%d d=%d)", who, B, d);
  if ((long)B * 3 * d > 0x7fffffffL) return set_error(M2_ERR_UNSUPPORTED, "%s: B * 3 d = %ld rows do not fit an int", who, (long)B * 3 * d);
  if (xproj_row < (long)B * L || xproj_row % 8)
    return set_error(M2_ERR_ARG, "%s: rows of xproj %ld apart, need a multiple of 8 from B * L = %ld on", who, xproj_row, (long)B * L);
  return launch_mixer_taps(xproj, xproj_row, u, short_w, short_b, proj_bias, FilterTaps{taps, skip_dev, nfilters}, y, B, L, d, (hipStream_t)stream);
}
