// Plans that a host thread keeps.  Planning walks tens to hundreds of tile shapes (1 us for an fp32 layer, 9 for an int8
// layer of 28x28 on the host, as long as the kernel it plans for), and a program plans the same few layers again and again:
// each thread keeps its last plans in a small table, the last four of those whose keys hash to one place (with one a place, two of
// a network's some fifty layers nearly always shared theirs, and were planned again at every call).
#pragma once
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>

namespace tsx {

// An environment variable that planners read, as a part of a plan's key (set but empty is another choice than not set); false
// where it is too long to be one.
struct PlanSwitch {
    char text[12];
    bool read(const char *name) {
        const char *value = std::getenv(name);
        if (!value) return true;
        if (std::strlen(value) + 2 > sizeof(text)) return false;
        text[0] = '=';
        std::strcpy(text + 1, value);
        return true;
    }
};

// The plan for `key`, a plain struct that was zeroed before it was filled, made by make() where it is not at hand.
template <class Plan, class Key, class Make>
Plan kept_plan(const Key &key, const Make &make) {
    constexpr int WAYS = 4, PLACES = 64;
    struct Place {
        Key keys[WAYS];
        Plan plans[WAYS];
        int used, next;      // entries; the oldest
    };
    static thread_local struct Table {
        Place *places = nullptr;
        ~Table() { delete[] places; places = nullptr; }
    } table;
    if (!table.places) table.places = new Place[PLACES]();
    static_assert(sizeof(Key) % sizeof(uint32_t) == 0, "the key is hashed by words");
    uint32_t h = 0;
    for (size_t i = 0; i < sizeof(Key) / sizeof(uint32_t); ++i) {
        uint32_t word;
        std::memcpy(&word, reinterpret_cast<const char *>(&key) + i * sizeof(word), sizeof(word));
        h = (h ^ word) * 0x9e3779b1u;
    }
    Place &place = table.places[h >> 26];
    for (int i = 0; i < place.used; ++i)
        if (std::memcmp(&place.keys[i], &key, sizeof(key)) == 0) return place.plans[i];
    const int at = place.next;
    place.plans[at] = make();
    place.keys[at] = key;
    place.next = (at + 1) % WAYS;
    if (place.used < WAYS) ++place.used;
    return place.plans[at];
}

}  // namespace tsx
