// Walks every address that a workgroup of the kernel for any size and alignment reads of a matrix contiguous along k, with
// the functions the kernel computes them with: each 16-byte load lies inside the tensor, and what is kept of it is what the
// product needs.  Prints the first case that does not hold and ends with 1.
#include <stdio.h>

#include <initializer_list>

#include "ptl_ragged_piece.hpp"

// A product's operand: `runs` matrices of rows x K, one behind the other; the slabs s0 .. s0 + ns - 1 of the tile at row r0.
template <int VEC>
static bool walk(int rows, int K, int runs, int r0, int s0, int ns) {
    constexpr int ES = 16 / VEC, SK = 8 * VEC, R = 32;
    const int per_run = (K + SK - 1) / SK, left = K - (per_run - 1) * SK;
    const long long row_b = (long long)K * ES, run_b = rows * row_b, bytes = runs * run_b;
    ptl::RagWalk w = {s0 % per_run, s0 / per_run, per_run, ns};
    long long base = w.run * run_b + r0 * row_b + w.pos * 128ll;
    for (int fetch = 0; fetch < ns + 2; ++fetch) {  // (the kernel asks for two more than it has)
        const unsigned want = w.want();
        const bool last = w.last();
        for (int pos = 0; pos < 8; ++pos) {
            const ptl::RagPiece q = ptl::rag_piece<VEC>(left, pos);
            for (int row = r0; row < r0 + R; ++row) {
                const long long at = base - (long long)ptl::RAG_AHEAD +
                                     ptl::rag_piece_at(ptl::rag_piece_off(row, r0, rows, (unsigned)row_b, pos), q.back, q.gap, last, want);
                bool ok = at >= 0 && at + 16 <= bytes;
                const long long mine = w.run * run_b + (row < rows ? row : rows - 1) * row_b;
                if (want) {
                    ok = ok && at >= mine && at + 16 <= mine + row_b;  // (inside the row: no other memory matters)
                    const int exist = !last ? VEC : q.tail <= 0 ? 0 : q.tail < VEC ? q.tail : VEC;
                    if (exist) ok = ok && at + (last ? q.cut : 0u) == mine + (w.pos * SK + pos * VEC) * (long long)ES;
                    if (exist) ok = ok && (last ? (int)q.cut : 0) == (VEC - exist) * ES;  // (zeros come in from above)
                }
                if (!ok) {
                    printf("VEC %d: %d runs of %d x %d, tile at row %d, slabs %d + %d: fetch %d, row %d, piece %d reads bytes "
                           "%lld .. %lld of %lld\n", VEC, runs, rows, K, r0, s0, ns, fetch, row, pos, at, at + 16, bytes);
                    return false;
                }
            }
        }
        if (w.next()) base = w.run * run_b + r0 * row_b + w.pos * 128ll;
    }
    return true;
}

template <int VEC>
static bool all() {
    constexpr int SK = 8 * VEC;
    for (int K = VEC; K <= 4 * SK + 1; ++K)
        for (int runs = 1; runs <= 3; runs += 2)
            for (int rows : {1, 31, 32, 33, 65}) {
                const int total = (K + SK - 1) / SK * runs;
                for (int r0 = 0; r0 < rows; r0 += 32)
                    for (int s0 = 0; s0 < total; ++s0)
                        for (int ns : {1, 2, total - s0})
                            if (s0 + ns <= total && !walk<VEC>(rows, K, runs, r0, s0, ns)) return false;
            }
    return true;
}

int main() { return all<4>() && all<8>() ? 0 : 1; }
