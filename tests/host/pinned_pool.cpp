// The pinned pool's chunks over the lives of the streams that read them.
#include <cstdio>
#include <cstdlib>

#include "pinned_pool.h"

using namespace nxm;

#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)

int main()
{
    constexpr size_t MB = 1u << 20;
    {
        auto pool = std::make_shared<PinnedPool>();
        Stream s;
        PendingUploads up;
        int a = -1, b = -1, c = -1, d = -1;
        char *pa = nullptr, *pb = nullptr, *pc = nullptr, *pd = nullptr;
        CHECK(pool->take(MB, &a, &pa) == hipSuccess);
        s.queued = 1;
        CHECK(up.add(pool, a, &s) == hipSuccess);
        // its copies are under way: another chunk, and the smallest free one that is enough
        CHECK(pool->take(3 * MB, &b, &pb) == hipSuccess && pb != pa);
        CHECK(up.poll() == hipSuccess);
        CHECK(pool->take(MB, &c, &pc) == hipSuccess && pc != pa && pc != pb);
        pool->give(b);
        pool->give(c);
        CHECK(pool->take(MB, &d, &pd) == hipSuccess && pd == pc);
        pool->give(d);
        // the stream is being captured: other threads take chunks all the same
        s.captured = true;
        CHECK(pool->take(MB, &d, &pd) == hipSuccess && pd == pc);
        pool->give(d);
        s.captured = false;
        // done, and seen to be
        s.done = 1;
        CHECK(up.poll() == hipSuccess);
        CHECK(pool->take(MB, &d, &pd) == hipSuccess && pd == pa);
        // queued again, and the stream goes with its world
        s.queued = 2;
        CHECK(up.add(pool, d, &s) == hipSuccess);
        CHECK(hipStreamSynchronize(&s) == hipSuccess);
        up.drain();
        s.gone = true;
        CHECK(pool->take(MB, &d, &pd) == hipSuccess && pd == pa);
        pool->give(d);
        CHECK(g_mallocs == 3 && g_events == 1);
    }
    CHECK(g_frees == 3 && g_events == 0);
    {
        // the context goes before the world that still has copies queued
        auto pool = std::make_shared<PinnedPool>();
        Stream s;
        PendingUploads up;
        int a = -1;
        char *pa = nullptr;
        CHECK(pool->take(MB, &a, &pa) == hipSuccess);
        s.queued = 1;
        CHECK(up.add(std::move(pool), a, &s) == hipSuccess);
        CHECK(g_frees == 3);
        s.done = 1;
        CHECK(up.poll() == hipSuccess && g_frees == 4);
        // a record that fails: waited for, and given back
        auto other = std::make_shared<PinnedPool>();
        CHECK(other->take(MB, &a, &pa) == hipSuccess);
        s.gone = true;
        CHECK(up.add(other, a, &s) != hipSuccess);
        char *again = nullptr;
        CHECK(other->take(MB, &a, &again) == hipSuccess && again == pa);
    }
    CHECK(g_frees == 5 && g_events == 0);
    std::printf("ok\n");
    return 0;
}
