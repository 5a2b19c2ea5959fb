// Checks of the kept tables (ciflow_amd/csrc/built_map.h) on the CPU: a table is
// made once per key, one whose construction throws is not kept, and what it had
// allocated until then goes back.  Built by tests/test_built_map.py.
#include "../../ciflow_amd/csrc/built_map.h"

#include <cstdio>
#include <cstdlib>
#include <memory>
#include <stdexcept>

#define CHECK(c)                                                    \
    do {                                                            \
        if (!(c)) {                                                 \
            std::printf("line %d: %s does not hold\n", __LINE__, #c); \
            std::exit(1);                                           \
        }                                                           \
    } while (0)

static int live = 0;
struct Part {
    Part() { ++live; }
    ~Part() { --live; }
};
struct Tables {  // two buffers, the second made last (move-only, as device buffers are)
    std::unique_ptr<Part> first, last;
};

int main() {
    std::map<std::pair<int, int>, Tables> m;
    const auto key = std::make_pair(12, 6);
    int made = 0;
    bool room = false;
    auto make = [&](Tables& t) {
        ++made;
        t.first.reset(new Part());
        if (!room) throw std::runtime_error("no memory");
        t.last.reset(new Part());
    };
    for (int i = 0; i < 2; ++i) {
        bool threw = false;
        try {
            cf::built_entry(m, key, make);
        } catch (const std::runtime_error&) {
            threw = true;
        }
        CHECK(threw && m.empty() && live == 0 && made == i + 1);  // tried again each time
    }
    room = true;
    Tables& t = cf::built_entry(m, key, make);
    CHECK(made == 3 && m.size() == 1 && t.first && t.last && live == 2);
    room = false;
    CHECK(&cf::built_entry(m, key, make) == &t && made == 3);
    bool threw = false;
    try {
        cf::built_entry(m, std::make_pair(12, 5), make);
    } catch (const std::runtime_error&) {
        threw = true;
    }
    CHECK(threw && m.size() == 1 && t.last);
    std::printf("all kept table checks passed\n");
    return 0;
}
