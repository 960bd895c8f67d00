// Plans that a host thread keeps.  Planning walks tens to hundreds of tile shapes (1 us for an fp32 layer, 9 for an int8
// layer of 28x28 on the host, as long as the kernel it plans for), and a program plans the same few layers again and again:
// each thread keeps its last plans, one per slot of a small table.
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
    struct Slot {
        Key key;
        bool used;
        Plan plan;
    };
    constexpr int SLOTS = 256;
    static thread_local struct Table {
        Slot *slots = nullptr;
        ~Table() { delete[] slots; slots = nullptr; }
    } table;
    if (!table.slots) table.slots = new Slot[SLOTS]();
    static_assert(sizeof(Key) % sizeof(uint32_t) == 0, "the key is hashed by words");
    uint32_t h = 0;
    for (size_t i = 0; i < sizeof(Key) / sizeof(uint32_t); ++i) {
        uint32_t word;
        std::memcpy(&word, reinterpret_cast<const char *>(&key) + i * sizeof(word), sizeof(word));
        h = (h ^ word) * 0x9e3779b1u;
    }
    Slot &slot = table.slots[h >> 24];
    if (!slot.used || std::memcmp(&slot.key, &key, sizeof(key)) != 0) {
        slot.plan = make();
        slot.key = key;
        slot.used = true;
    }
    return slot.plan;
}

}  // namespace tsx
