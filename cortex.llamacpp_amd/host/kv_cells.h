// kv_cells.h — the cells of the KV cache as the host knows them, and the sums over their chunks that searches of the table go by.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace mi355 {

struct KVCell {
    int32_t pos = -1;                  // < 0: free
    int32_t delta = 0;
    uint64_t seqs = 0;
};

// What every chunk of 64 cells holds.  A search for a sequence's cells, or for a free one, passes over the chunks that have none: a server's cache has thousands of cells and a tick looks for one
// of each conversation.  Sixteen conversations in 8.9 k cells, us a tick before the device has anything to do: their last tokens taken back 56, cells found 36, chunk lists 8 cell by cell.
// A chunk's sum is made anew by the first search that needs it after one of its cells has changed (touch).
class CellChunks {
  public:
    struct Sum {
        uint64_t seqs = 0;             // sequences of its occupied cells
        int32_t max_pos = -1, used = 0;
    };
    void reset(size_t n_cells) { sums_.assign((n_cells + 63) / 64, Sum()); stale_.assign(sums_.size(), 0); }
    void touch(int cell) { stale_[(size_t)cell >> 6] = 1; }
    const Sum &at(const std::vector<KVCell> &cells, int chunk) {
        Sum &s = sums_[(size_t)chunk];
        if (stale_[(size_t)chunk]) {
            s = Sum();
            for (size_t i = (size_t)chunk * 64, e = std::min(cells.size(), i + 64); i < e; i++)
                if (cells[i].pos >= 0) { s.seqs |= cells[i].seqs; s.max_pos = std::max(s.max_pos, cells[i].pos); s.used++; }
            stale_[(size_t)chunk] = 0;
        }
        return s;
    }
    // f(i) for every cell i < end, in order, but for those of chunks without a cell at position p0 or behind it (or, seqs not 0, without one of these sequences); f may change cell i
    template <class F> void each(const std::vector<KVCell> &cells, int end, uint64_t seqs, int p0, F f) {
        for (int i = 0; i < end; i += 64) {
            const Sum &s = at(cells, i >> 6);
            if (s.used == 0 || s.max_pos < p0 || (seqs != 0 && (s.seqs & seqs) == 0)) continue;
            for (int j = i, e = std::min(end, i + 64); j < e; j++) f(j);
        }
    }
    // the lowest free cell of [lo, hi) that is not taken[], -1: none
    template <class T> int first_free(const std::vector<KVCell> &cells, int lo, int hi, const T &taken) {
        for (int i = lo; i < hi;) {
            if ((i & 63) == 0 && i + 64 <= hi && at(cells, i >> 6).used == 64) { i += 64; continue; }
            if (cells[(size_t)i].pos < 0 && !taken[(size_t)i]) return i;
            i++;
        }
        return -1;
    }

  private:
    std::vector<Sum> sums_;
    std::vector<uint8_t> stale_;
};

}  // namespace mi355
