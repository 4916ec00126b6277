// The sliced ELL plan written out plainly on the host: what the device's
// (sell_plan.hip) has to equal.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

#include "../../fluidity_amd/csrc/krylov_common.h"

namespace flgpu {

// Host-side plan of a sliced ELL operand: slot offsets, column indices
// (int16 offsets from the slice's first row, or its window's, when they all
// fit) and, per slot, the entry of the source value array it takes (vmap[k]
// for CSR entry k, or k itself; -1 for padding); the slices' rows when
// sorted; the offsets and masks of diagonal slices.
struct SellHost {
    int nsl = 0;
    int64_t nslot = 0;
    bool use16 = false;
    std::vector<int32_t> sptr, src, c32, rows, off;
    std::vector<int16_t> c16;
    std::vector<uint64_t> mask;
    double fill(int64_t nnz) const { return nnz > 0 ? (double)nslot / (double)nnz : 1.0; }
};

// The distinct offsets col - row of the given rows, ascending, if there are
// at most `most` of them and each row's columns ascend.
inline bool sell_offsets(const int32_t* rowptr, const int32_t* col, const int32_t* rows, int nr, int most,
                         std::vector<int32_t>& off) {
    off.clear();
    std::vector<int32_t> merged;
    for (int q = 0; q < nr; q++) {
        const int r = rows[q], len = rowptr[r + 1] - rowptr[r];
        const int32_t* c = col + rowptr[r];
        bool same = len == (int)off.size();
        for (int j = 0; same && j < len; j++) same = c[j] - r == off[j];
        if (same) continue;
        for (int j = 1; j < len; j++)
            if (c[j] <= c[j - 1]) return false;
        merged.clear();
        size_t a = 0;
        for (int j = 0; j < len; j++) {
            while (a < off.size() && off[a] < c[j] - r) merged.push_back(off[a++]);
            if (a < off.size() && off[a] == c[j] - r) a++;
            merged.push_back(c[j] - r);
        }
        merged.insert(merged.end(), off.begin() + a, off.end());
        if ((int)merged.size() > most) return false;
        off.swap(merged);
    }
    return true;
}

inline void sell_plan(const int32_t* rowptr, const int32_t* col, int n, const int32_t* vmap, SellHost& h,
                      int window = 0, bool diagonals = false, int run = 0) {
    diagonals = diagonals && rowptr[n] < 1 << 30;  // (their extra steps keep within 32-bit slots)
    h.nsl = (n + kSlice - 1) / kSlice;
    h.rows.clear();
    h.off.clear();
    h.mask.clear();
    if (window) {
        h.rows.assign((size_t)h.nsl * kSlice, -1);
        for (int r = 0; r < n; r++) h.rows[r] = r;
        if (!run) run = window;
        for (int w0 = 0; w0 < n; w0 += run)
            std::stable_sort(h.rows.begin() + w0, h.rows.begin() + std::min(n, w0 + run),
                             [&](int32_t a, int32_t b) { return rowptr[a + 1] - rowptr[a] > rowptr[b + 1] - rowptr[b]; });
    }
    auto row_of = [&](int sl, int lane) {
        const int q = sl * kSlice + lane;
        return window ? h.rows[q] : q < n ? q : -1;
    };
    auto first = [&](int sl) { return window ? sl * kSlice / window * window : sl * kSlice; };
    h.sptr.assign((size_t)h.nsl + 1, 0);
    std::vector<int32_t> alloff;  // the diagonal slices' offsets, one after the other
    std::vector<uint8_t> dia(h.nsl, 0);
    std::vector<int32_t> off;
    for (int sl = 0; sl < h.nsl; sl++) {
        int w = 0, nr = 0;
        int32_t rows[kSlice];
        for (int lane = 0; lane < kSlice; lane++) {
            const int r = row_of(sl, lane);
            if (r < 0) continue;
            rows[nr++] = r;
            w = std::max(w, rowptr[r + 1] - rowptr[r]);
        }
        if (diagonals && sell_offsets(rowptr, col, rows, nr, w + w / 8, off)) {
            dia[sl] = 1;
            w = (int)off.size();
            alloff.insert(alloff.end(), off.begin(), off.end());
        }
        h.sptr[sl + 1] = h.sptr[sl] + w * kSlice;
    }
    h.nslot = h.sptr[h.nsl];
    h.src.assign((size_t)h.nslot, -1);
    // the columns' width first, so that only one array is written
    bool fits = true;
    for (int sl = 0; fits && sl < h.nsl; sl++) {
        const int r0 = first(sl);
        for (int lane = 0; !dia[sl] && lane < kSlice; lane++) {
            const int r = row_of(sl, lane);
            if (r < 0) continue;
            bool far = r - r0 > 32767;  // (its padding's column)
            for (int k = rowptr[r]; k < rowptr[r + 1]; k++) far |= col[k] - r0 < -32768 || col[k] - r0 > 32767;
            fits = fits && !far;
        }
    }
    h.use16 = fits;
    h.c16.assign(fits ? (size_t)h.nslot : 0, 0);
    h.c32.assign(fits ? 0 : (size_t)h.nslot, 0);
    if (!alloff.empty()) h.off.assign((size_t)h.nslot / kSlice + kSellAhead, 0);
    h.mask.assign((size_t)h.nslot / kSlice + kSellAhead, 0);
    size_t at = 0;
    for (int sl = 0; sl < h.nsl; sl++) {
        const int r0 = first(sl), w = (h.sptr[sl + 1] - h.sptr[sl]) / kSlice;
        if (dia[sl]) {
            const size_t g = (size_t)h.sptr[sl] / kSlice;
            for (int j = 0; j < w; j++) h.off[g + j] = alloff[at + j];
            at += w;
            for (int lane = 0; lane < kSlice; lane++) {
                const int r = row_of(sl, lane);
                if (r < 0) continue;
                int j = 0;
                for (int k = rowptr[r]; k < rowptr[r + 1]; k++) {
                    while (h.off[g + j] != col[k] - r) j++;
                    h.src[(g + j) * kSlice + lane] = vmap ? vmap[k] : k;
                    h.mask[g + j] |= (uint64_t)1 << lane;
                }
            }
            continue;
        }
        for (int lane = 0; lane < kSlice; lane++) {
            const int r = row_of(sl, lane);
            const int len = r >= 0 ? rowptr[r + 1] - rowptr[r] : 0;
            for (int j = 0; j < w; j++) {
                const size_t slot = (size_t)h.sptr[sl] + (size_t)j * kSlice + lane;
                int cj = r >= 0 ? r : r0;
                if (j < len) {
                    const int k = rowptr[r] + j;
                    h.src[slot] = vmap ? vmap[k] : k;
                    h.mask[slot / kSlice] |= (uint64_t)1 << lane;
                    cj = col[k];
                }
                if (fits)
                    h.c16[slot] = (int16_t)(cj - r0);
                else
                    h.c32[slot] = cj;
            }
        }
    }
    for (int sl = 0; sl < h.nsl; sl++) h.sptr[sl] |= dia[sl];
}

}  // namespace flgpu
