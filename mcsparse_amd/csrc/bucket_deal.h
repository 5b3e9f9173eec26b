// How the groups of runs of a crowded bucket are dealt to the workgroups that share it (spmv_transposed.hip).
#ifndef MCSPARSE_AMD_BUCKET_DEAL_H_
#define MCSPARSE_AMD_BUCKET_DEAL_H_

#include <cstdint>

namespace mcsp {

// Wavefront w of every part walks the groups w, w + waves, ... and adds those that are its part's.  The parts take turns
// along that walk, so every wavefront of every part gets its share (dealt by g % parts a wavefront would meet the same
// part all along its walk wherever parts and waves have a common factor, and most wavefronts would add nothing); the
// wavefronts begin with different parts, so that buckets of few groups, one to a wavefront, are spread as well.
// A transposing call on 100 M nonzeros in a million columns, one bucket of 4 and of 8 times the mean: 550 and 602 us dealt
// by g % parts, 499 and 497 us so (no crowded bucket: 430); on 33 M 198 and 219, 182 and 183 (158).
constexpr uint32_t part_of_group(uint32_t group, uint32_t waves, uint32_t parts) {
    return (group / waves + group % waves) % parts;
}

}  // namespace mcsp

#endif  // MCSPARSE_AMD_BUCKET_DEAL_H_
