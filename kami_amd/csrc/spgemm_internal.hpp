// Structure phase of C = A * B in two launches, for callers of the library that allocate C
// themselves; not part of the public interface.
#pragma once
#include "../../include/kami.h"

// Block rows of A it takes: the workgroup of every row sums all rows' counts.
constexpr int32_t kStructureRows = 4096;

// kami_bsr_spgemm_symbolic and _fill in one call.  colidxC holds `capacity` entries; with
// nnzb(C) above that (returned all the same) it is not written and kami_bsr_spgemm_fill has
// to follow.  ws holds the symbolic workspace and A->mb int32 counts after it
// (KAMI_ENOSPC below that); KAMI_ENOTSUP above kStructureRows.
extern "C" kami_status kami_bsr_spgemm_structure(const kami_bsr* A, const kami_bsr* B, int32_t* rowptrC,
                                                 int32_t* colidxC, int64_t capacity, int64_t* nnzbC,
                                                 void* ws, size_t ws_bytes, void* stream);
