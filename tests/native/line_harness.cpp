// Host build of the line filter (test infrastructure): the cell-pair engine's
// filter of one probe against one staging slot.
#include "../../nanofiller_amd/csrc/nf_line.h"

extern "C" {

// probe, slot: 8 floats (x y z cx cy cz l a), centres from the common origin.
// Writes the filter's value (negative: the pair goes on) for the lines and for
// every pair within reach.
void nfh_slot_apart(const float* probe, const float* slot, int valid, float R_max, float ew, float S, float out[2]) {
  const float4 D1 = make_float4(probe[3], probe[4], probe[5], probe[7]);
  const float4 D2 = make_float4(slot[3], slot[4], slot[5], slot[7]);
  const float hl1 = 0.5f * probe[6], hl2 = 0.5f * slot[6];
  const nf::LineFilter f = nf::line_filter(R_max, ew, S);
  const nf::LineSide l = nf::line_side(f, probe[0], probe[1], probe[2], D1);
  out[0] = nf::slot_apart<false>(make_float4(l.ux, l.uy, l.uz, l.mx), make_float2(l.my, l.mz),
                                 nf::slot_side<false>(f, slot[0], slot[1], slot[2], hl2, D2, valid != 0));
  const float x = probe[0], y = probe[1], z = probe[2];
  const float rp = (hl1 * 1.000001f + (R_max + 16.0f * ew)) * 1.000006f, slack = 64.0f * nf::U32 * S * S;
  out[1] = nf::slot_apart<true>(make_float4(2.0f * x, 2.0f * y, 2.0f * z, 2.0f * rp),
                                make_float2(fmaf(z, z, fmaf(y, y, x * x)) - fmaf(rp, rp, slack), 0.0f),
                                nf::slot_side<true>(f, slot[0], slot[1], slot[2], hl2, D2, valid != 0));
}

}  // extern "C"
