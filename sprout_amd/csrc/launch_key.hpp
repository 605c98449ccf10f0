// Keys of captured launches: the bytes of everything a captured kernel holds
// by value or by address.  A graph is replayed only for an equal key.
#pragma once

#include <cstdint>
#include <vector>

namespace mi {

using Launch_key = std::vector<uint8_t>;

// (values without padding)
template <class... T>
void put_key(Launch_key& key, T const&... values) {
    auto const put = [&key](auto const& v) {
        uint8_t const* b = reinterpret_cast<uint8_t const*>(&v);
        key.insert(key.end(), b, b + sizeof(v));
    };
    (put(values), ...);
}

}  // namespace mi
