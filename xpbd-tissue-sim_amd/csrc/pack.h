// Objects of a batch into tiles.
#pragma once
#include <cstddef>
#include <cstdint>
#include <vector>

namespace xpbd {

// The tile of each of n objects, in order: an object joins the last one's tile where
// each of its m loads (load[m * object + k]) fits in with what limit[k] leaves, else it
// starts the next.
inline std::vector<int32_t> pack_objects(int n, const std::vector<int64_t>& load, const std::vector<int64_t>& limit)
{
    const size_t m = limit.size();
    std::vector<int64_t> held(m, 0);
    std::vector<int32_t> tile(n);
    int32_t t = 0;
    for (int i = 0; i < n; i++) {
        bool fits = true;
        for (size_t k = 0; k < m; k++) fits = fits && held[k] + load[m * i + k] <= limit[k];
        if (!fits && i > 0) {
            t++;
            held.assign(m, 0);
        }
        for (size_t k = 0; k < m; k++) held[k] += load[m * i + k];
        tile[i] = t;
    }
    return tile;
}

}  // namespace xpbd
