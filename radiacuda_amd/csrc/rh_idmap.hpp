// rh_idmap.hpp -- ids of the vertices, edges and faces of a mesh (host packing).
#pragma once

#include <array>
#include <cstdint>
#include <cstring>
#include <vector>

namespace rh {

// Ids of vertices, edges and faces in order of first occurrence:
// open addressing over a table of ids at most half full, keys stored in id
// order (no allocation per key).  The key's words are mixed by a multiplication
// each, and the slot is taken from the upper half of a last product: a
// multiplication moves bits upwards only, and the coordinates of a regular grid
// differ in their highest bits alone (from the lower half, a row of 1,000 boxes
// of 40 x 20 x 5 mm shared 16 slots: 630 probes a vertex).  Models are packed on
// every geometry change, so this is on the path of a gradient step: 1,000
// polyhedra of an undulator take 2.1 ms of one core of either kind, regular or
// random sizes, where ordered maps and a vector per face took 13 ms on a slower
// one (a step over them 12.8 -> 7.8 ms).
using VKey = std::array<uint64_t, 3>;   // bits of the coordinates
using EKey = std::array<int32_t, 2>;    // ascending vertex ids
using FKey = std::array<int32_t, 4>;    // ascending vertex ids, a triangle's first one -1
inline VKey vkey(const double* v)
{
    VKey k;
    std::memcpy(k.data(), v, 3 * sizeof(double));
    return k;
}
inline uint64_t mix(uint64_t h, uint64_t w)
{
    h = (h ^ w) * 0x9E3779B97F4A7C15ull;
    return h ^ (h >> 29);
}
// The last mixing: the upper half of a product, which every bit below reaches,
// after the high bits have been folded down.
inline uint64_t spread(uint64_t h) { return ((h ^ (h >> 32)) * 0x9E3779B97F4A7C15ull) >> 32; }
inline uint64_t word2(int32_t a, int32_t b) { return (uint64_t(uint32_t(a)) << 32) | uint32_t(b); }
inline uint64_t hash_key(const VKey& k) { return mix(mix(mix(1, k[0]), k[1]), k[2]); }
inline uint64_t hash_key(const EKey& k) { return mix(1, word2(k[0], k[1])); }
inline uint64_t hash_key(const FKey& k) { return mix(mix(1, word2(k[0], k[1])), word2(k[2], k[3])); }

template <class Key>
class IdMap {
public:
    explicit IdMap(size_t expect)
    {
        keys_.reserve(expect);
        size_t n = 16;
        while (n < 2 * expect) n *= 2;
        slot_.assign(n, -1);
    }
    // id of the key, a new one if it is not there
    int32_t add(const Key& k)
    {
        size_t i = place(k);
        if (slot_[i] >= 0) return slot_[i];
        if (2 * (keys_.size() + 1) > slot_.size()) {
            slot_.assign(2 * slot_.size(), -1);
            for (size_t q = 0; q < keys_.size(); q++) slot_[place(keys_[q])] = int32_t(q);
            i = place(k);
        }
        keys_.push_back(k);
        return slot_[i] = int32_t(keys_.size() - 1);
    }
    int32_t find(const Key& k) const { return slot_[place(k)]; }
    size_t size() const { return keys_.size(); }
    const Key& operator[](size_t id) const { return keys_[id]; }

    // mean number of slots looked at to find a key that is there
    double probes() const
    {
        const size_t m = slot_.size() - 1;
        double n = 0.0;
        for (const Key& k : keys_) n += double(1 + ((place(k) - home(k, m)) & m));
        return keys_.empty() ? 0.0 : n / double(keys_.size());
    }

private:
    static size_t home(const Key& k, size_t m) { return size_t(spread(hash_key(k))) & m; }
    size_t place(const Key& k) const
    {
        const size_t m = slot_.size() - 1;
        size_t i = home(k, m);
        while (slot_[i] >= 0 && keys_[size_t(slot_[i])] != k) i = (i + 1) & m;
        return i;
    }
    std::vector<Key> keys_;
    std::vector<int32_t> slot_;
};

}  // namespace rh
