// Launches of the grouped expert qmm for large buckets (dspark_moe_wide.h).
#include <algorithm>

#include "dspark_moe_wide.h"

namespace dspark {
namespace {

template <int BITS, int MT, int NT, bool PW>
void launch_mode(const wide::MoeWideArgs& a, bool swiglu, hipStream_t s) {
  const dim3 grid((unsigned)a.per_xcd * 8), block(wide::kThreads);
  if (swiglu) hipLaunchKernelGGL((wide::moe_wide_kernel<BITS, MT, NT, PW, true>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((wide::moe_wide_kernel<BITS, MT, NT, PW, false>), grid, block, 0, s, a);
}

template <int BITS, int MT>
void launch_form(const wide::MoeWideArgs& a, bool swiglu, bool packed, hipStream_t s) {
  if (packed) launch_mode<BITS, MT, 4, true>(a, swiglu, s);
  else launch_mode<BITS, MT, 4, false>(a, swiglu, s);
}

}  // namespace

// Row tile of a workgroup / 16, by the rows of a bucket on average. 32 rows leave room for three
// workgroups per CU; 64 rows unpack a weight once for twice the rows. Measured (block of 128 experts,
// top 8, 2048 x 768, 4 bits): 32 rows a bucket 196 us against 220, 62 rows 268 against 285; 8 bits:
// 32 rows 235 / 236, 62 rows 325 / 300; 64 experts, 2048 x 1024, 4 bits: 125 rows 258 / 251. 16 and
// 48 rows were no better anywhere (32 rows a bucket: 218 and 217 us).
int moe_wide_mt(long P, long E, int bits) { return P >= (bits == 8 ? 60 : 112) * E ? 4 : 2; }

// This kernel reads an expert's weights once for 32 or 64 rows, where the small-bucket kernels take 4
// rows a pass and 16 a workgroup; but its K loop is one workgroup's, so a call takes 25 us and 0.55 us
// for every 64 of H and of I whatever the rows, which few pairs through few or small experts do not pay.
// Fitted to 6570 calls through both (4 to 256 experts, top 1 to 8, 512 x 256 to 4096 x 1536, packed and
// row-major, 0.5 to 40 rows an expert): 26 of them take this kernel and are more than 3% slower for it,
// the worst 1.16 times. Small-bucket / this, us, 4 bits: 128 experts top 8, 2048 x 768, 64 tokens 125 / 132,
// 96 tokens 157 / 133; 8 experts top 2 of that size, 64 tokens 54 / 56, 128 tokens 61 / 58; 64 experts top 8,
// 512 x 256, 48 tokens 25 / 36, 128 tokens 51 / 39. H past 2048 takes the small-bucket kernels' slowest form
// (16 experts top 2, 4096 x 1536, 48 tokens: 150 / 89).
bool moe_wide(long M, long H, long I, long E, long k, int bits) {
  if (M <= 16) return false;
  const double pairs = (double)M * k, size = 1e-6 * H * I;
  if (H > 2048) return pairs * size >= (bits == 8 ? 50 : 250);
  // the small-bucket launches also grow with the experts and with the rows a bucket could hold
  const double few = std::min({(bits == 8 ? 300 : 450) / size, 32768.0 / E, 256.0 * k});
  return pairs >= std::max({few, (3 + 0.375 * k) * E, 1024.0 / E});
}

template <int BITS>
void launch_rows(const wide::MoeWideArgs& a, bool swiglu, bool packed, int mt, hipStream_t s) {
  if (mt == 2) launch_form<BITS, 2>(a, swiglu, packed, s);
  else launch_form<BITS, 4>(a, swiglu, packed, s);
}

int launch_moe_wide(wide::MoeWideArgs a, bool swiglu, bool packed, int mt, int bits, hipStream_t s) {
  a.strips = (a.N + (swiglu ? 127 : 255)) / (swiglu ? 128 : 256);
  const long items = (long)a.max_tiles * a.strips;
  if (items > (1L << 30)) return fail(DSPARK_ERR_SHAPE, "moe_switch_glu: too many tiles");
  a.per_xcd = (int)((items + 7) / 8);
  if (bits == 8) launch_rows<8>(a, swiglu, packed, mt, s);
  else launch_rows<4>(a, swiglu, packed, mt, s);
  return check_launch(swiglu ? "moe gate/up" : "moe down");
}

}  // namespace dspark
