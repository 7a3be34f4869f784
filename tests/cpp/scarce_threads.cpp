// The threads that help with large results are not needed: without them, or
// without memory to make them, the calls return the same results.
//   scarce_threads pages         Prefault alone, on the CPU
//   scarce_threads gpu           whole solves
// This program's pthread_create and operator new stand in for the C library's
// (it is linked with -rdynamic) and fail on demand.
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>
#include <sys/mman.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <thread>
#include <vector>

#include "../../include/sssp_mi355x.h"

static std::atomic<int> g_threads_left{1 << 30};  // pthread_create calls that still succeed
static std::atomic<int> g_news_left{1 << 30};

extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *x)
{
    typedef int (*Fn)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    static const Fn real = (Fn)dlsym(RTLD_NEXT, "pthread_create");
    if (g_threads_left.fetch_sub(1) <= 0) return EAGAIN;
    return real(t, a, f, x);
}

void *operator new(size_t n)
{
    if (g_news_left.fetch_sub(1) <= 0) throw std::bad_alloc();
    if (void *p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

namespace sssp {
class Prefault {  // sssp_graph.hpp
  public:
    Prefault(void *dst, size_t bytes);
    ~Prefault();
    void join();

  private:
    static constexpr int kThreads = 8;
    std::atomic<bool> go_{false};
    std::thread threads_[kThreads];
    int n_ = 0;
};
}  // namespace sssp

static int pages()
{
    const size_t bytes = (size_t)300 << 20;
    for (int what = 0; what < 2; what++)
        for (int left = 0; left < 12; left++) {
            void *m = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
            if (m == MAP_FAILED) return 1;
            std::printf("%s: %d succeed\n", what ? "operator new" : "pthread_create", left);
            std::fflush(stdout);
            (what ? g_news_left : g_threads_left) = left;
            {
                sssp::Prefault p(m, bytes);
                g_news_left = g_threads_left = 1 << 30;
                if (left % 2) p.join();
            }
            for (size_t i = 0; i < bytes; i += 1 << 20)
                if (((char *)m)[i] != 0) return 1;
            munmap(m, bytes);
        }
    std::printf("pages ok\n");
    return 0;
}

#define CHECK(call)                                                    \
    do {                                                               \
        if ((call) != SSSP_OK) {                                       \
            std::printf("%s: %s\n", #call, sssp_last_error());         \
            return 1;                                                  \
        }                                                              \
    } while (0)

static int gpu()
{
    // 3 M vertices: results of 12 MB (distances) and 3 MB (flags)
    const int32_t V = 3000000;
    std::vector<int32_t> src, dst;
    std::vector<float> w;
    for (int32_t v = 0; v < V; v += 3) {
        src.push_back(0);
        dst.push_back(v);
        w.push_back((float)(v % 1000));
    }
    std::vector<float> want((size_t)V), got((size_t)V);
    for (int left : {0, 1, 3, 1 << 30}) {  // a first graph each: the threads are made anew
        sssp_graph *g = nullptr;
        CHECK(sssp_graph_create(SSSP_W_F32, src.data(), dst.data(), w.data(), V,
                                (int64_t)src.size(), 0, SSSP_NO_CSC, &g));
        CHECK(sssp_solve(g, 0, SSSP_SCHED_HEURISTIC, nullptr, nullptr));  // the runtime's own threads
        std::printf("solve with %d threads to be had\n", left);
        std::fflush(stdout);
        std::memset(got.data(), 0, 4 * (size_t)V);
        g_threads_left = left;
        CHECK(sssp_solve(g, 0, SSSP_SCHED_HEURISTIC, got.data(), nullptr));
        CHECK(sssp_get_distances(g, got.data()));
        g_threads_left = 1 << 30;
        CHECK(sssp_graph_destroy(g));
        for (int32_t v = 0; v < V; v++)
            if (got[(size_t)v] != (v % 3 ? 3.402823466e38f : (float)(v % 1000))) {
                std::printf("vertex %d: %g\n", v, got[(size_t)v]);
                return 1;
            }
    }
    std::printf("gpu ok\n");
    return 0;
}

int main(int argc, char **argv)
{
    return argc > 1 && std::strcmp(argv[1], "gpu") == 0 ? gpu() : pages();
}
