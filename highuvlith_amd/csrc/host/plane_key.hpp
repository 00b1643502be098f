// Keys of what a context keeps per plane list (kernel stacks, pointer tables,
// recorded launches), and their removal when a kernel set dies.
#pragma once

#include <algorithm>
#include <cstdint>
#include <utility>
#include <vector>

namespace huvi {

// The ids of a plane list apart from the numbers that tell its entries apart
// (sizes, layout flags): an id is never compared with one of those.
struct PlaneKey {
  std::vector<uint64_t> ksets;
  std::vector<uint64_t> form;
  bool operator<(const PlaneKey& o) const {
    return ksets != o.ksets ? ksets < o.ksets : form < o.form;
  }
};

// Erases the entries whose key holds set `id`; drop(value) frees each first.
template <class Map, class Drop>
void forget_entries(Map& map, uint64_t id, Drop drop) {
  for (auto it = map.begin(); it != map.end();) {
    const std::vector<uint64_t>& k = it->first.ksets;
    if (std::find(k.begin(), k.end(), id) == k.end()) {
      ++it;
    } else {
      drop(it->second);
      it = map.erase(it);
    }
  }
}

}  // namespace huvi
