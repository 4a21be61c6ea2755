/* mgx::hold (mgx_call_buffer.h) over an allocator that has so much memory and no more */
#include "mgx_call_buffer.h"

#include <cstdio>
#include <map>

static std::map<unsigned char *, size_t> blocks;
static size_t room = 0, used = 0, allocs = 0, frees = 0;

static unsigned char *take(size_t n)
{
    allocs++;
    if (used + n > room) return nullptr;
    unsigned char *p = new unsigned char[1];
    blocks[p] = n;
    used += n;
    return p;
}

static void give(unsigned char *p)
{
    frees++;
    used -= blocks.at(p);
    blocks.erase(p);
    delete[] p;
}

static int failures = 0;
#define CHECK(x)                                             \
    do {                                                     \
        if (!(x)) {                                          \
            std::printf("line %d: %s\n", __LINE__, #x);      \
            failures++;                                      \
        }                                                    \
    } while (0)

int main()
{
    using mgx::Held;
    unsigned char *p = nullptr;
    size_t bytes = 0;
    const auto hold = [&](size_t needed, size_t extra) {
        allocs = frees = 0;
        return mgx::hold(p, bytes, needed, extra, take, give);
    };

    /* the extra bytes do not fit: the needed ones are held, and later calls free nothing */
    room = 100;
    CHECK(hold(40, 80) == Held::Needed && p && bytes == 40 && used == 40);
    for (int i = 0; i < 3; i++) {
        unsigned char *before = p;
        CHECK(hold(40, 80) == Held::Needed && p == before && bytes == 40);
        CHECK(frees == 0 && allocs == 1);
    }
    /* a smaller call takes what is there */
    CHECK(hold(30, 10) == Held::All && allocs == 0);
    CHECK(hold(30, 0) == Held::All && allocs == 0);
    /* memory has come back */
    room = 200;
    CHECK(hold(40, 80) == Held::All && bytes == 120 && used == 120 && frees == 1);
    /* more of both: beside the old one they do not fit, after it they do */
    CHECK(hold(130, 60) == Held::All && bytes == 190 && used == 190 && frees == 1);
    /* more than there is: the needed bytes alone */
    CHECK(hold(195, 60) == Held::Needed && bytes == 195 && used == 195);
    /* nothing fits: no buffer, and the next call that fits gets one */
    CHECK(hold(300, 0) == Held::None && !p && bytes == 0 && used == 0);
    CHECK(hold(50, 10) == Held::All && bytes == 60);
    CHECK(used == 60 && blocks.size() == 1);
    std::printf(failures ? "failed\n" : "ok\n");
    return failures != 0;
}
