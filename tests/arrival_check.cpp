// Host check of the arrival count (cudallm_amd/csrc/arrival.h): in every order in which the members of a call can take
// their steps, from any content of the word, exactly one of them is last, and it comes after all shares are published.
// The calls below run one after the other on the word that the one before left, some with the tag of an earlier one.
//
//   arrival_check      prints "ok" and the number of orders, or what went wrong, and exits 1
#include <cstdio>
#include <cstdlib>
#include <random>
#include <set>
#include <vector>

#include "arrival.h"

using namespace cllm;

namespace {

struct Word {
    uint64_t* p;
    void compare_exchange(uint64_t from, uint64_t to) const {
        if (*p == from) *p = to;
    }
    uint64_t add_one() const { return (*p)++; }
    void store(uint64_t v) const { *p = v; }
};

struct Member {
    int step = 0;  // 0 see, 1 begin, 2 publish, 3 arrive, 4 done
    uint64_t seen = 0;
};

struct State {
    uint64_t word;
    std::vector<Member> m;
    int published = 0, lasts = 0;
};

void fail(const char* what, uint64_t start) {
    std::printf("%s, from a word of %016llx\n", what, static_cast<unsigned long long>(start));
    std::exit(1);
}

void take_step(State& s, size_t i, uint64_t tag, uint64_t start) {
    Member& m = s.m[i];
    const Word w{&s.word};
    switch (m.step++) {
        case 0: m.seen = s.word; break;
        case 1: arrival::begin(w, m.seen, tag); break;
        case 2: ++s.published; break;
        case 3:
            if (arrival::arrive(w, tag, static_cast<unsigned>(s.m.size()))) {
                ++s.lasts;
                if (s.published != static_cast<int>(s.m.size())) fail("last before all shares were published", start);
            }
            break;
    }
}

void check_end(const State& s, uint64_t start) {
    if (s.lasts != 1) fail(s.lasts ? "more than one last" : "no last", start);
    if (s.word != 0) fail("a count left behind", start);
}

long orders = 0;
void every_order(const State& s, uint64_t tag, uint64_t start) {
    bool any = false;
    for (size_t i = 0; i < s.m.size(); ++i)
        if (s.m[i].step < 4) {
            State t = s;
            take_step(t, i, tag, start);
            every_order(t, tag, start);
            any = true;
        }
    if (!any) {
        ++orders;
        check_end(s, start);
    }
}

}  // namespace

int main() {
    const uint64_t salt = 0x1234567890abcdefull, tag = arrival::tag_of(salt, 0), other = arrival::tag_of(salt, 1);
    const uint64_t starts[] = {0, ~0ull, 0xFFC00000FFC00000ull, 0x7FC000007FC00000ull, 0xFFC00000FFFFFFFFull, 0x3F8000003F800000ull,
                               0xDEADBEEFDEADBEEFull, 1, 255, other, other | 1, other | 2, other | 255};
    for (uint64_t start : starts)
        for (size_t n = 2; n <= 3; ++n) every_order(State{start, std::vector<Member>(n)}, tag, start);

    // More members, in orders drawn at random, on the word of the call before; every third call repeats an earlier tag.
    std::mt19937_64 rng(7);
    uint64_t word = 0xFFC00000FFC00000ull;
    for (int call = 0; call < 3000; ++call) {
        if (call % 5 == 4) word = rng();
        const uint64_t start = word, t = arrival::tag_of(salt, call % 3 == 2 ? call / 2 : call);
        State s{word, std::vector<Member>(2 + rng() % 63)};
        std::vector<size_t> open(s.m.size());
        for (size_t i = 0; i < open.size(); ++i) open[i] = i;
        while (!open.empty()) {
            const size_t k = rng() % open.size(), i = open[k];
            take_step(s, i, t, start);
            if (s.m[i].step == 4) open[k] = open.back(), open.pop_back();
        }
        ++orders;
        check_end(s, start);
        word = s.word;
    }

    // Tags: no two alike, none that a fill or the usual NaNs hold.
    for (uint64_t sl : {uint64_t{0}, salt, ~uint64_t{0}}) {
        std::set<uint64_t> seen;
        for (uint64_t n = 0; n < 200000; ++n) seen.insert(arrival::tag_of(sl, n));
        if (seen.size() != 200000) fail("two calls with one tag", sl);
        for (uint64_t w : {~uint64_t{0}, uint64_t{0xFFC00000FFC00000}, uint64_t{0x7FC000007FC00000}})
            if (seen.count(w & ~arrival::kCount)) fail("a tag that memory holds", w);
    }
    std::printf("ok %ld\n", orders);
    return 0;
}
