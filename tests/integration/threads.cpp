// parallel_for and WorkerPool where the system starts no more threads after the
// first `room`: the work runs on those there are.  pthread_create here stands
// before libc's for the whole process.
#include <dlfcn.h>
#include <pthread.h>

#include <atomic>
#include <cstdio>
#include <vector>

#include "og_internal.h"

static std::atomic<int> room{1 << 20};

extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
    if (room.fetch_sub(1) <= 0) return 11;  // EAGAIN
    using Fn = int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    return ((Fn)dlsym(RTLD_NEXT, "pthread_create"))(t, a, f, arg);
}

static int bad = 0;
static void check(bool ok, const char *what, int threads) {
    if (!ok) {
        printf("%s with %d threads\n", what, threads);
        bad = 1;
    }
}

int main() {
    for (int n : {0, 1, 3, 100}) {
        room = n;
        std::vector<std::atomic<int>> seen(1000);
        og::parallel_for(1000, 7, 5, [&](uint64_t b, uint64_t e, unsigned) {
            for (uint64_t i = b; i < e; ++i) seen[i]++;
        });
        for (auto &x : seen) check(x == 1, "parallel_for", n);
        room = n;
        og::WorkerPool pool(4);
        const unsigned want = 1 + (n < 3 ? n : 3);
        check(pool.size() == want, "size", n);
        for (int k = 0; k < 3; ++k) {
            std::atomic<unsigned> calls{0}, ids{0};
            pool.run([&](unsigned t) {
                calls++;
                ids |= 1u << t;
            });
            check(calls == want && ids == (1u << want) - 1, "run", n);
        }
    }
    return bad;
}
