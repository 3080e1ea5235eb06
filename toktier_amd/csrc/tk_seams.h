// tk_seams.h -- host side of the seam tables (tk_device.h): what the symbols
// of a rule table spell, and the tables of what they hold across each of
// their inner positions. Built once when an engine opens.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <utility>
#include <vector>

#include "tk_device.h"

namespace tk {

// What each symbol spells, by id (tk_engine_open takes ids below 2^20), all in
// one buffer; len 0: nothing.
struct Spelled {
  std::vector<uint8_t> bytes;
  std::vector<uint32_t> at;
  std::vector<uint16_t> len;
  bool is(uint64_t id, const uint8_t* s, size_t n) const {
    return id < len.size() && len[id] == n && !std::memcmp(bytes.data() + at[id], s, n);
  }
};

// The strings of the bytes and of every rule's product (from the rules alone:
// product = left + right). False when they are not plain (a byte without an
// id, an id with two spellings, a string over MAX_LEN bytes or over MAX_TOTAL
// bytes of them, far above any vocabulary: they bound the memory that opening
// a table takes): the engine then looks for no seams. A rule whose sides no
// byte sequence reaches never runs and spells nothing.
inline bool symbol_strings(const uint64_t* keys, const uint64_t* vals, uint64_t count,
                           const int32_t* byte_id, Spelled& sp) {
  constexpr size_t MAX_LEN = 4096, MAX_TOTAL = (size_t)32 << 20, MAX_IDS = 1u << 20;
  auto put = [&](uint64_t id, size_t at, size_t n) {
    if (id >= sp.len.size()) {
      sp.at.resize(id + 1);
      sp.len.resize(id + 1);
    }
    if (sp.len[id]) {  // known: the same string, or not plain
      const bool same = sp.is(id, sp.bytes.data() + at, n);
      sp.bytes.resize(at);
      return same;
    }
    sp.at[id] = (uint32_t)at;
    sp.len[id] = (uint16_t)n;
    return at + n <= MAX_TOTAL;
  };
  for (int b = 0; b < 256; ++b) {
    const size_t at = sp.bytes.size();
    sp.bytes.push_back((uint8_t)b);
    if (byte_id[b] < 0 || (size_t)byte_id[b] >= MAX_IDS ||
        !put((uint64_t)byte_id[b], at, 1)) return false;
  }
  // the rules in rank order (each rule has its own rank; one that shares it
  // comes last, which costs a pass)
  struct Rule { uint32_t l, r, id; };
  constexpr uint32_t NONE = ~0u;
  std::vector<Rule> todo, later;
  for (uint64_t i = 0; i < count; ++i) {
    if (keys[i] == ~0ULL) continue;
    const uint64_t rank = vals[i] >> 32;
    const Rule u{(uint32_t)(keys[i] >> 32), (uint32_t)keys[i], (uint32_t)vals[i]};
    if (rank >= MAX_IDS || u.l >= MAX_IDS || u.r >= MAX_IDS || u.id >= MAX_IDS) return false;
    if (rank >= todo.size()) todo.resize(rank + 1, Rule{NONE, 0, 0});
    if (todo[rank].l == NONE) todo[rank] = u;
    else later.push_back(u);
  }
  todo.insert(todo.end(), later.begin(), later.end());
  // (in rank order nearly every rule's sides are known by its turn)
  for (size_t left = todo.size() + 1; todo.size() < left && !todo.empty();) {
    left = todo.size();
    later.clear();
    for (const Rule& u : todo) {
      if (u.l == NONE) continue;  // (a rank without a rule)
      if (u.l >= sp.len.size() || u.r >= sp.len.size() || !sp.len[u.l] || !sp.len[u.r]) {
        later.push_back(u);
        continue;
      }
      const size_t at = sp.bytes.size(), nl = sp.len[u.l], nr = sp.len[u.r];
      if (nl + nr > MAX_LEN) return false;
      sp.bytes.resize(at + nl + nr);
      std::memcpy(sp.bytes.data() + at, sp.bytes.data() + sp.at[u.l], nl);
      std::memcpy(sp.bytes.data() + at + nl, sp.bytes.data() + sp.at[u.r], nr);
      if (!put(u.id, at, nl + nr)) return false;
    }
    todo.swap(later);
  }
  return true;
}

// The seam tables (tk_device.h) of those strings, and of `more` (the
// vocabulary entries that no symbol spells, for tables with a whole-piece
// rule): every inner position of every string, as its byte pair's key type and
// its key. The bitmap has 16 bits or more per byte of the strings, up to 2^24 (2 MB).
struct SeamTables {
  std::vector<uint16_t> mask;
  std::vector<uint32_t> bits;
  uint32_t shift = 0;
};
inline void build_seams(const Spelled& sp,
                        const std::vector<std::pair<const uint8_t*, size_t>>& more,
                        SeamTables& t) {
  size_t total = sp.bytes.size();
  for (const auto& s : more) total += s.second;
  uint32_t lg = 16;
  while (lg < 24 && ((size_t)1 << lg) < 16 * total) ++lg;
  t.mask.assign(65536, 0);
  t.bits.assign((size_t)1 << (lg - 5), 0);
  t.shift = 32 - lg;
  auto add = [&](const uint8_t* p, size_t n) {
    uint32_t left = 0;  // the bytes before, nearest lowest
    for (size_t i = 1; i < n; ++i) {
      left = left << 8 | p[i - 1];
      const size_t A = std::min<size_t>(i, SEAM_CTX), B = std::min<size_t>(n - i, SEAM_CTX);
      uint32_t right = 0;
      for (size_t k = 0; k < B; ++k) right |= (uint32_t)p[i + k] << (8 * k);
      const uint32_t type = (uint32_t)((A - 1) * SEAM_CTX + (B - 1));
      t.mask[(size_t)p[i - 1] << 8 | p[i]] |= (uint16_t)(1u << type);
      const uint32_t h = seam_hash(left, right, type) >> t.shift;
      t.bits[h >> 5] |= 1u << (h & 31);
    }
  };
  static_assert(SEAM_CTX == 4, "left holds four bytes");
  for (size_t id = 0; id < sp.len.size(); ++id)
    if (sp.len[id] > 1) add(sp.bytes.data() + sp.at[id], sp.len[id]);
  for (const auto& s : more) add(s.first, s.second);
}

}  // namespace tk
