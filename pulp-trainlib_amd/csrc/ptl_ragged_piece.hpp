// Which bytes a workgroup of the kernel for any size and alignment (ptl_ragged.inc) reads of a matrix that is contiguous
// along k: plain C++ for the host and the device, so that a test can walk every address on the CPU.
#pragma once

#ifdef __HIP__
#define PTL_BOTH __host__ __device__
#else
#define PTL_BOTH
#endif

namespace ptl {

// A thread's piece of VEC elements at position `pos` (0 .. 7) of a slab, where the last slab of a run has `left` elements.
// Every load has its 16 bytes inside the run, which holds at least one piece:
//   * a piece that reaches over the end of the run is read so that it ENDS there and shifted down by `cut`;
//   * one that does not exist is read from the last slab's first k - or, where that slab itself is shorter than a piece,
//     from the run's last one (`gap`) - and replaced by zeros.
struct RagPiece {
    int tail;       // elements from the piece's first k on in the last slab
    unsigned gap;   // bytes that the last slab lacks of one piece
    unsigned back;  // bytes that the piece is read earlier in the last slab (at least `gap`)
    unsigned cut;   // bytes
};
template <int VEC>
PTL_BOTH inline RagPiece rag_piece(int left, int pos) {
    constexpr unsigned ES = 16 / VEC;
    RagPiece r;
    r.tail = left - pos * VEC;
    r.gap = left < VEC ? (unsigned)(VEC - left) * ES : 0u;
    r.cut = r.tail > 0 && r.tail < VEC ? (unsigned)(VEC - r.tail) * ES : 0u;
    r.back = r.tail <= 0 ? (unsigned)pos * 16u + r.gap : r.cut;
    return r;
}
// Offsets are counted from a piece before the slab, so that they are never negative: a scalar address and 32 bits a lane.
constexpr unsigned RAG_AHEAD = 16;
// Of the piece at `pos` of a row, from the start of row r0 of the slab; rows beyond the end repeat the last one.
PTL_BOTH inline unsigned rag_piece_off(int row, int r0, int rows, unsigned row_b, int pos) {
    return ((unsigned)(row < rows ? row : rows - 1) - (unsigned)r0) * row_b + (unsigned)pos * 16u + RAG_AHEAD;
}
// Where it is read.  want: nothing is needed any more where this is 0, every lane reads the same piece.
PTL_BOTH inline unsigned rag_piece_at(unsigned off, unsigned back, unsigned gap, bool last, unsigned want) {
    return want ? off - (last ? back : 0u) : RAG_AHEAD - (last ? gap : 0u);
}

// The slabs of a workgroup in order: position in their run, and the run.  A workgroup asks for more slabs than it has, so
// that every step waits for the same number of loads: behind the last one the walk stands still and `want` is 0.
struct RagWalk {
    int pos, run, per_run, left;
    PTL_BOTH inline bool last() const { return pos + 1 == per_run; }
    PTL_BOTH inline unsigned want() const { return left > 0 ? ~0u : 0u; }
    // On to the next slab, if there is one.
    PTL_BOTH inline bool next() {
        if (--left <= 0) return false;
        const bool end = last();
        pos = end ? 0 : pos + 1;
        run += end ? 1 : 0;
        return true;
    }
};

}  // namespace ptl
