// The codec's host copy where no thread, the first one only, or every thread can be made (g++ -Wl,--wrap=pthread_create).
#include <cerrno>
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
    for (int threads : {0, 1, 2, 1 << 30})
        for (size_t bytes : {(size_t)0, (size_t)1, ((size_t)1 << 20) - 1, (size_t)1 << 20, ((size_t)1 << 20) + 1, ((size_t)3 << 20) + 4097, ((size_t)4 << 20) + 3}) {
            std::vector<unsigned char> src(bytes + 1), dst(bytes + 64, 0xA5);
            for (size_t i = 0; i < bytes; i++) src[i] = (unsigned char)(i * 2654435761u >> 13);
            g_left = threads;
            pmh::CopyTeam().copy(dst.data(), src.data(), bytes);
            for (size_t i = 0; i < bytes; i++)
                if (dst[i] != src[i]) return std::printf("threads %d bytes %zu: differs at %zu\n", threads, bytes, i), 1;
            for (size_t i = bytes; i < dst.size(); i++)
                if (dst[i] != 0xA5) return std::printf("threads %d bytes %zu: written past the end\n", threads, bytes), 1;
        }
    return 0;
}
