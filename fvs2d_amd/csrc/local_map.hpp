// Local index of a cell or node in a block (keys: id | periodic shift << 27).
#pragma once
#include <cstddef>
#include <vector>

namespace fvs {

// open addressing, at most half full: a node of many cells may bring any number
// of keys before its block is found not to fit
class LocalMap {
  std::vector<unsigned> key = std::vector<unsigned>(256, ~0u);
  std::vector<int> val = std::vector<int>(256);
  std::vector<size_t> used;

  size_t slot(unsigned k) const {
    size_t h = (k * 2654435761u >> 8) & (key.size() - 1);
    while (key[h] != ~0u && key[h] != k) h = (h + 1) & (key.size() - 1);
    return h;
  }
  void grow() {
    std::vector<unsigned> k0(2 * key.size(), ~0u);
    std::vector<int> v0(k0.size());
    k0.swap(key);
    v0.swap(val);
    for (size_t &h : used) {
      const size_t g = slot(k0[h]);
      key[g] = k0[h];
      val[g] = v0[h];
      h = g;
    }
  }

 public:
  void clear() {
    for (size_t h : used) key[h] = ~0u;
    used.clear();
  }
  size_t size() const { return used.size(); }
  // the entry of k, created (fresh) if there is none; valid until the next call
  int &at(unsigned k, bool &fresh) {
    size_t h = slot(k);
    fresh = key[h] == ~0u;
    if (fresh) {
      if (2 * used.size() >= key.size()) {
        grow();
        h = slot(k);
      }
      key[h] = k;
      used.push_back(h);
    }
    return val[h];
  }
};

}  // namespace fvs
