// The seam tables' host build (tk_seams.h) as a library for the CPU tests.
#include "../toktier_amd/csrc/tk_seams.h"

// 0: no seams; else the bitmap's shift, with the mask (65,536 entries) and
// the bitmap's words (at most 2^19) copied out, and the number of words
extern "C" int seam_tables(const uint64_t* keys, const uint64_t* vals, uint64_t count,
                           const int32_t* byte_id, uint16_t* mask, uint32_t* bits,
                           uint64_t* words) {
  tk::Spelled sp;
  if (!tk::symbol_strings(keys, vals, count, byte_id, sp)) return 0;
  tk::SeamTables t;
  tk::build_seams(sp, {}, t);
  std::copy(t.mask.begin(), t.mask.end(), mask);
  std::copy(t.bits.begin(), t.bits.end(), bits);
  *words = t.bits.size();
  return (int)t.shift;
}
