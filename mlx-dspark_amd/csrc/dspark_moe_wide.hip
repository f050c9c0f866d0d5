// Launches of the grouped expert qmm for large buckets (dspark_moe_wide.h).
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
