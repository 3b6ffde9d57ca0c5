// One team for many copies, one after the other, with every number of helpers that can be made (g++ -Wl,--wrap=pthread_create).
#include <cerrno>
#include <chrono>
#include <cstdio>
#include <vector>

#include "../../pmetal_amd/csrc/host_copy.hpp"

static int g_left = 1 << 30;  // threads that can still be made
extern "C" int __real_pthread_create(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
extern "C" int __wrap_pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
    if (g_left-- <= 0) return EAGAIN;
    return __real_pthread_create(t, a, f, arg);
}

int main() {
    const size_t k = (size_t)1 << 10;
    for (int threads : {0, 1, 2, 1 << 30}) {
        g_left = threads;
        pmh::CopyTeam team;
        for (int round = 0; round < 60; round++)
            for (size_t bytes : {(size_t)0, (size_t)1, 128 * k - 1, 128 * k, 128 * k + 1, 256 * k + 3, 1024 * k + 4097}) {
                std::vector<unsigned char> src(bytes + 1), dst(bytes + 64, 0xA5);
                for (size_t i = 0; i < bytes; i++) src[i] = (unsigned char)((i + (size_t)round) * 2654435761u >> 13);
                if (round % 20 == 19) std::this_thread::sleep_for(std::chrono::milliseconds(2));  // the helpers sleep by now
                team.copy(dst.data(), src.data(), bytes);
                if (bytes && memcmp(dst.data(), src.data(), bytes)) return std::printf("threads %d round %d bytes %zu: differs\n", threads, round, bytes), 1;
                for (size_t i = bytes; i < dst.size(); i++)
                    if (dst[i] != 0xA5) return std::printf("threads %d round %d bytes %zu: written past the end\n", threads, round, bytes), 1;
            }
    }
    return 0;
}
