// tk_seams.h -- host side of the seam tables (tk_device.h): what the symbols
// of a rule table spell, and the tables of what they hold across each of
// their inner positions. Built once when an engine opens.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <string>
#include <utility>
#include <vector>

#include "tk_device.h"

namespace tk {

// The strings that a symbol can spell: the bytes of every rule's product
// (from the rules alone: product = left + right) and, for tables with a
// whole-piece rule, the vocabulary entries. False when they are not plain
// (a byte without an id, an id with two spellings, a string over MAX_LEN bytes
// or over MAX_TOTAL bytes of them, far above any vocabulary: they bound the
// memory that opening a table takes): the engine then looks for no seams. A
// rule whose sides no byte sequence reaches never runs and spells nothing.
inline bool symbol_strings(const uint64_t* keys, const uint64_t* vals, uint64_t count,
                           const int32_t* byte_id, std::vector<std::string>& out) {
  constexpr size_t MAX_LEN = 4096, MAX_TOTAL = (size_t)32 << 20;
  size_t total = 0;
  std::vector<std::string> of;  // by id (tk_engine_open takes ids below 2^20)
  auto put = [&](uint64_t id, std::string s) {
    if (id >= of.size()) of.resize(id + 1);
    if (of[id].empty()) of[id] = std::move(s);
    else if (of[id] != s) return false;
    return true;
  };
  for (int b = 0; b < 256; ++b)
    if (byte_id[b] < 0 || !put((uint64_t)byte_id[b], std::string(1, (char)b))) return false;
  struct Rule { uint64_t rank, l, r, id; };
  std::vector<Rule> todo;
  for (uint64_t i = 0; i < count; ++i)
    if (keys[i] != ~0ULL)
      todo.push_back({vals[i] >> 32, keys[i] >> 32, keys[i] & 0xFFFFFFFFULL,
                      vals[i] & 0xFFFFFFFFULL});
  std::sort(todo.begin(), todo.end(),
            [](const Rule& a, const Rule& b) { return a.rank < b.rank; });
  // (in rank order nearly every rule's sides are known by its turn)
  for (size_t left = todo.size() + 1; todo.size() < left && !todo.empty();) {
    left = todo.size();
    std::vector<Rule> later;
    for (const Rule& u : todo) {
      if (u.l >= of.size() || u.r >= of.size() || of[u.l].empty() || of[u.r].empty()) {
        later.push_back(u);
        continue;
      }
      std::string s = of[u.l] + of[u.r];
      if (s.size() > MAX_LEN || (total += s.size()) > MAX_TOTAL || !put(u.id, s))
        return false;
      out.push_back(std::move(s));
    }
    todo.swap(later);
  }
  return true;
}

// The seam tables (tk_device.h) of those strings: every inner position of
// every string, as its byte pair's key type and its key. The bitmap has at
// least 16 bits per key, up to 2^24 (2 MB).
struct SeamTables {
  std::vector<uint16_t> mask;
  std::vector<uint32_t> bits;
  uint32_t shift = 0;
};
inline void build_seams(const std::vector<std::string>& strings, SeamTables& t) {
  size_t keys = 0;
  for (const std::string& s : strings) keys += s.size();
  uint32_t lg = 16;
  while (lg < 24 && ((size_t)1 << lg) < 8 * keys) ++lg;  // (half the keys repeat)
  t.mask.assign(65536, 0);
  t.bits.assign((size_t)1 << (lg - 5), 0);
  t.shift = 32 - lg;
  for (const std::string& s : strings) {
    const uint8_t* p = reinterpret_cast<const uint8_t*>(s.data());
    for (size_t i = 1; i < s.size(); ++i) {
      const int A = (int)std::min<size_t>(i, SEAM_CTX);
      const int B = (int)std::min<size_t>(s.size() - i, SEAM_CTX);
      uint32_t left = 0, right = 0;
      for (int k = 0; k < A; ++k) left |= (uint32_t)p[i - 1 - k] << (8 * k);
      for (int k = 0; k < B; ++k) right |= (uint32_t)p[i + k] << (8 * k);
      const uint32_t type = (uint32_t)((A - 1) * SEAM_CTX + (B - 1));
      t.mask[(size_t)p[i - 1] << 8 | p[i]] |= (uint16_t)(1u << type);
      const uint32_t h = seam_hash(left, right, type) >> t.shift;
      t.bits[h >> 5] |= 1u << (h & 31);
    }
  }
}

}  // namespace tk
