// Tables made once per key and kept (a context's shape tables): an entry is in
// the map only once it is complete, so that one whose construction threw is
// made again by the next call instead of being used half made.
//
// No HIP in this file: it is tested on the CPU with tables of its own.
#pragma once

#include <map>
#include <utility>

namespace cf {

// The entry of `key`; make(Value&) fills a new one, and what it throws leaves
// the map as it was.
template <class Key, class Value, class Make>
Value& built_entry(std::map<Key, Value>& m, const Key& key, Make&& make) {
    const auto it = m.find(key);
    if (it != m.end()) return it->second;
    Value v;
    make(v);
    return m.emplace(key, std::move(v)).first->second;
}

}  // namespace cf
