// Word of a face record (DevMesh::rec): bit 31 set on a boundary face; bit 30,
// the record's own side is the reference owner's; bits 0-29, the record of
// the face's other side, or the boundary face.
//
// Records have a bit more than cells (NBR_INDEX_MASK): a cell has up to four,
// so a mesh of 2^29 cells can have more than 2^29 (in the input order of the
// library's own boxes 1.2 to 1.4 per cell).  Contexts with more than REC_MAX of
// them keep the sweeps that gather per lane.
#pragma once
#include <cstdint>

#include "physics.hpp"

namespace nf {

constexpr uint32_t REC_BOUNDARY = 0x80000000u, REC_OWNER = 0x40000000u, REC_INDEX_MASK = 0x3FFFFFFFu;
constexpr uint64_t REC_MAX = (uint64_t)REC_INDEX_MASK + 1;  // records that can be numbered

NF_HD uint32_t rec_word(bool boundary, bool owner, uint32_t index) {
    return (boundary ? REC_BOUNDARY : 0u) | (owner ? REC_OWNER : 0u) | index;
}
NF_HD uint32_t rec_index(uint32_t w) { return w & REC_INDEX_MASK; }

}  // namespace nf
