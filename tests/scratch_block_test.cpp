// Drives jitnn_amd/csrc/scratch.h with an allocator that keeps books (no GPU).  Prints the name of each check; exit status 0: all hold.
#include <cstdio>
#include <cstdlib>
#include <map>

#include "scratch.h"

static std::map<void *, size_t> live;  // address -> bytes
static size_t room = (size_t)1 << 40;  // bytes the "device" has
static bool refuse_release = false;
static int asked = 0;

struct BookMem {
    static size_t used() {
        size_t u = 0;
        for (auto &b : live) u += b.second;
        return u;
    }
    static void *alloc(size_t bytes) {
        ++asked;
        if (used() + bytes > room) return nullptr;
        static size_t next = 0x1000;
        void *p = (void *)next;
        next += bytes;
        live[p] = bytes;
        return p;
    }
    static bool release(void *p) {
        if (refuse_release) return false;
        if (!live.erase(p)) abort();  // freed twice
        return true;
    }
};
using Block = jitnn::ScratchBlock<BookMem>;
constexpr size_t MiB = (size_t)1 << 20;

#define CHECK(e)                                                       \
    do {                                                               \
        if (!(e)) {                                                    \
            printf("%s:%d: %s does not hold\n", __FILE__, __LINE__, #e); \
            exit(1);                                                   \
        }                                                              \
    } while (0)

static void fresh() {
    live.clear();
    room = (size_t)1 << 40;
    refuse_release = false;
    asked = 0;
}

static void grows_and_reuses() {
    fresh();
    Block b;
    bool waited = false;
    void *p = b.get(3 * MiB + 1, false, &waited);
    CHECK(p && b.capacity() == 4 * MiB && !waited);
    CHECK(b.get(4 * MiB, false, &waited) == p && b.growths() == 1);
    void *q = b.get(5 * MiB, false, &waited);
    CHECK(q && q != p && waited && live.size() == 1 && live.count(q) && b.retired_bytes() == 0);
    b.release_all();
    CHECK(live.empty() && b.capacity() == 0);
}

// A graph records an address; a later eager call needs more.  The recorded block must still be allocated, and new work must
// not be given it.
static void recorded_block_outlives_growth() {
    fresh();
    Block b;
    bool waited = false;
    void *p = b.get(32 * MiB, false, &waited);
    CHECK(b.get(32 * MiB, true, &waited) == p);  // recorded
    void *q = b.get(150 * MiB, false, &waited);
    CHECK(q && q != p && !waited && live.count(p) && live.count(q) && b.retired_bytes() == 32 * MiB);
    CHECK(b.get(32 * MiB, false, &waited) == q);
    void *r = b.get(200 * MiB, false, &waited);  // q was never recorded
    CHECK(r && waited && !live.count(q) && live.count(p));
    b.release_all();
    CHECK(live.empty() && b.retired_bytes() == 0);
}

// Recording at every size: what is kept for graphs stays below what is in use.
static void retired_blocks_are_bounded() {
    fresh();
    Block b;
    bool waited = false;
    for (size_t s = 1; s <= 300; ++s) {
        CHECK(b.get(s * MiB, true, &waited));
        CHECK(b.retired_bytes() < b.capacity());
    }
    b.release_all();
    CHECK(live.empty());
    // where twice the size is not to be had, what the call needs is enough
    room = 100 * MiB;
    CHECK(b.get(40 * MiB, true, &waited) && b.get(60 * MiB, false, &waited));
    CHECK(b.capacity() == 60 * MiB && b.retired_bytes() == 40 * MiB);
    b.release_all();
    CHECK(live.empty());
}

// An address that the runtime would not take back (a capture forbids it) is kept too, and given back later.
static void refused_release_is_not_lost() {
    fresh();
    Block b;
    bool waited = false;
    void *p = b.get(MiB, false, &waited);
    refuse_release = true;
    void *q = b.get(2 * MiB, false, &waited);
    CHECK(q && q != p && !waited && live.size() == 2);
    refuse_release = false;
    b.release_all();
    CHECK(live.empty());
}

// A call that can do without: refused, it keeps what is there, and does not ask for that size or a larger one again.
static void refused_growth_keeps_the_block() {
    fresh();
    Block b;
    bool waited = false;
    void *p = b.try_get(10 * MiB, false, &waited);
    CHECK(p);
    room = 50 * MiB;
    CHECK(!b.try_get(45 * MiB, false, &waited) && live.count(p) && b.capacity() == 10 * MiB && !waited);
    const int before = asked;
    CHECK(!b.try_get(45 * MiB, false, &waited) && !b.try_get(60 * MiB, false, &waited) && asked == before);
    CHECK(b.try_get(10 * MiB, false, &waited) == p && asked == before);
    CHECK(b.try_get(20 * MiB, false, &waited) && asked == before + 1 && waited);  // smaller than what was refused
    room = 200 * MiB;
    CHECK(!b.try_get(45 * MiB, false, &waited) && asked == before + 1);
    b.ask_again();
    CHECK(b.try_get(45 * MiB, false, &waited) && asked == before + 2);
    CHECK(b.try_get(45 * MiB, true, &waited) && !b.try_get(60 * MiB, true, &waited) && asked == before + 2);  // no growth under a capture
    b.release_all();
    room = 10 * MiB;
    CHECK(!b.try_get(11 * MiB, false, &waited));
    b.release_all();  // forgets the refusal
    room = 20 * MiB;
    CHECK(b.try_get(11 * MiB, false, &waited));
    b.release_all();
    CHECK(live.empty());
}

// A prompt pass asks again for what was refused, also one whose launches need nothing ahead (a prompt of few tokens).
static void a_pass_asks_again() {
    fresh();
    Block operands, weights;
    bool waited = false;
    room = 10 * MiB;
    CHECK(!operands.try_get(11 * MiB, false, &waited) && !weights.try_get(12 * MiB, false, &waited));
    room = 100 * MiB;
    const int before = asked;
    CHECK(!operands.try_get(11 * MiB, false, &waited) && !weights.try_get(12 * MiB, false, &waited) && asked == before);
    jitnn::start_pass(operands, weights, 0, 0, &waited);
    CHECK(asked == before && operands.try_get(11 * MiB, false, &waited) && weights.try_get(12 * MiB, false, &waited));
    jitnn::start_pass(operands, weights, 20 * MiB, 30 * MiB, &waited);
    CHECK(operands.capacity() == 20 * MiB && weights.capacity() == 30 * MiB && waited);
    room = 60 * MiB;
    jitnn::start_pass(operands, weights, 40 * MiB, 0, &waited);  // no room: the block stays
    CHECK(operands.capacity() == 20 * MiB && live.size() == 2);
    operands.release_all();
    weights.release_all();
    CHECK(live.empty());
}

// A call that cannot do without gives up the old block where there is no room for both, but never one a graph may hold.
static void needed_growth_gives_up_the_block() {
    fresh();
    Block b;
    bool waited = false;
    room = 50 * MiB;
    CHECK(b.get(30 * MiB, false, &waited) && b.get(40 * MiB, false, &waited) && waited && b.capacity() == 40 * MiB && live.size() == 1);
    CHECK(!b.get(60 * MiB, false, &waited));
    CHECK(b.get(30 * MiB, true, &waited) && !b.get(40 * MiB, false, &waited) && live.size() == 1 && b.capacity() == 30 * MiB);
    CHECK(!b.give_up(&waited));
    b.release_all();
    CHECK(live.empty() && !b.give_up(&waited));
}

int main() {
#define RUN(f) (f(), printf(#f "\n"))
    RUN(grows_and_reuses);
    RUN(recorded_block_outlives_growth);
    RUN(retired_blocks_are_bounded);
    RUN(refused_release_is_not_lost);
    RUN(refused_growth_keeps_the_block);
    RUN(a_pass_asks_again);
    RUN(needed_growth_gives_up_the_block);
    return 0;
}
