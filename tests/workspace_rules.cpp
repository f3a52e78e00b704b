// The workspace's growth rules on the host: a pretend memory of so many floats, and a count of
// what was asked of it. Prints the first rule broken and exits with 1.
#include <cstdio>
#include <map>
#include <set>

#include "eb_workspace.h"

struct Mem {
    size_t room;
    std::map<float *, size_t> held;
    std::set<float *> gone;
    int allocs = 0, drains = 0;
    char *next = nullptr;
    eb_status alloc(size_t floats, float **p) {
        ++allocs;
        if (floats > room) return EB_OUT_OF_MEMORY;
        room -= floats;
        next += 64;
        *p = reinterpret_cast<float *>(next);
        held[*p] = floats;
        return EB_OK;
    }
    eb_status drain() { return ++drains, EB_OK; }
    eb_status free(float *p) {
        if (!held.count(p)) return EB_OTHER;
        room += held[p];
        held.erase(p);
        gone.insert(p);
        return EB_OK;
    }
};

static int line = 0;
#define RULE(x) do { if (!(x) && !line) { line = __LINE__; std::printf("line %d: %s\n", line, #x); } } while (0)

int main() {
    {  // plain growth: the old buffer goes after a drain; no growth, nothing asked
        eb::Workspace w;
        Mem m{1000};
        RULE(w.grow(m, 100, 100) == EB_OK && w.floats() == 100 && m.drains == 0);
        float *p = w.ptr();
        RULE(w.grow(m, 100, 10) == EB_OK && w.ptr() == p && m.allocs == 1);
        RULE(w.grow(m, 950, 950) == EB_OK && w.floats() == 950 && m.drains == 1);  // no room for both
        RULE(m.gone.count(p) && m.held.size() == 1 && m.room == 50);
        RULE(w.grow(m, 2000, 2000) == EB_OUT_OF_MEMORY && w.ptr() == nullptr && w.floats() == 0);
        w.free_all(m);
        RULE(m.held.empty() && m.room == 1000);
    }
    {  // less would do: what holds it is kept when memory is refused, without a drain
        eb::Workspace w;
        Mem m{1000};
        RULE(w.grow(m, 600, 600) == EB_OK);
        float *p = w.ptr();
        RULE(w.grow(m, 700, 20) == EB_OK && w.ptr() == p && w.floats() == 600 && m.drains == 0);
        RULE(m.allocs == 2);
        for (int i = 0; i < eb::kRefusedCalls; ++i) RULE(w.grow(m, 700 + i, 20) == EB_OK);
        RULE(m.allocs == 2 && w.ptr() == p);                         // refused: not asked again at once
        RULE(w.grow(m, 700, 20) == EB_OK && m.allocs == 3);          // but now and then
        m.room = 5000;
        RULE(w.grow(m, 650, 20) == EB_OK && w.floats() == 650);      // a smaller size is tried
        RULE(w.grow(m, 700, 20) == EB_OK && w.floats() == 650);      // (a larger one is still refused)
        for (int i = 0; i < eb::kRefusedCalls; ++i) RULE(w.grow(m, 700, 20) == EB_OK);
        RULE(w.floats() == 700);                                     // until it is asked for again
        RULE(w.grow(m, 800, 20) == EB_OK && w.floats() == 800);      // and then at once
        RULE(m.held.size() == 1);
    }
    {  // nothing there yet: least alone
        eb::Workspace w;
        Mem m{100};
        RULE(w.grow(m, 700, 20) == EB_OK && w.floats() == 20);
        RULE(w.grow(m, 700, 30) == EB_OK && w.floats() == 30);
        RULE(w.grow(m, 700, 130) == EB_OUT_OF_MEMORY);
    }
    {  // a graph keeps the buffer it was captured with, through both kinds of growth
        eb::Workspace w;
        Mem m{1000};
        RULE(w.ref() == nullptr);
        RULE(w.grow(m, 100, 100) == EB_OK);
        float *a = w.ref();
        RULE(w.ref() == a);
        RULE(w.grow(m, 200, 50) == EB_OK && m.drains == 0 && m.held.count(a));
        float *b = w.ref();
        RULE(w.grow(m, 300, 300) == EB_OK && m.held.size() == 3);
        w.unref(m, a);
        RULE(m.held.count(a));
        w.unref(m, a);
        RULE(!m.held.count(a) && m.held.count(b));
        float *c = w.ref();
        w.unref(m, c);
        RULE(m.held.count(c) && w.ptr() == c);                       // the current one stays
        w.free_all(m);
        RULE(m.held.empty());
    }
    return line ? 1 : 0;
}
