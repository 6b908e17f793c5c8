/* transfer CPUS: Transfer::to_host on a stream that is busy for 0.4 s, with the process held to CPUS cores (0: all).
   Prints: threads of the process, CPU seconds of the first copy, whether all copies were right, whether a failing
   copy was reported. */
#include <dirent.h>
#include <sched.h>
#include <sys/resource.h>

#include <cstdio>

#include "../../spacetime-optics_amd/csrc/transfer.h"

static double cpu_s() {
    rusage u;
    getrusage(RUSAGE_SELF, &u);
    return u.ru_utime.tv_sec + u.ru_stime.tv_sec + 1e-6 * (u.ru_utime.tv_usec + u.ru_stime.tv_usec);
}

static int threads() {
    int n = 0;
    DIR* d = opendir("/proc/self/task");
    while (dirent* e = readdir(d)) n += e->d_name[0] != '.';
    closedir(d);
    return n;
}

int main(int, char** argv) {
    const int cpus = std::atoi(argv[1]);
    if (cpus > 0) {
        cpu_set_t all, some;
        sched_getaffinity(0, sizeof all, &all);
        CPU_ZERO(&some);
        for (int i = 0, n = 0; i < CPU_SETSIZE && n < cpus; ++i)
            if (CPU_ISSET(i, &all)) CPU_SET(i, &some), ++n;
        sched_setaffinity(0, sizeof some, &some);
    }
    auto t = Transfer::of_device(0);
    bool right = true;
    double first = -1.0;
    const size_t M = size_t(1) << 20;
    for (size_t n : {3 * M, size_t(1), Transfer::MIN_BYTES - 1, Transfer::MIN_BYTES, 3 * M + 5, 16 * M, 16 * M + 4097, 70 * M + 1}) {
        std::vector<unsigned char> src(n), dst(n + 1, 77);
        for (size_t i = 0; i < n; ++i) src[i] = (unsigned char)(i * 2654435761u >> 13);
        const double c0 = cpu_s();
        if (first < 0) stub::busy_ms = 400;
        right = t->to_host(dst.data(), src.data(), n, nullptr) == hipSuccess && right;
        if (first < 0) first = cpu_s() - c0;
        right = right && std::memcmp(dst.data(), src.data(), n) == 0 && dst[n] == 77;
    }
    // the first, a later, and the last of its pieces fails; the next copy is right again
    bool reported = true;
    for (int k : {0, 2, 17}) {
        std::vector<unsigned char> src(70 * M, 5), dst(70 * M, 6);
        const size_t before = stub::copies;
        stub::fail_at = (long)before + k;
        const hipError_t e = t->to_host(dst.data(), src.data(), src.size(), nullptr);
        reported = (e != hipSuccess) == (stub::copies > before + (size_t)k) && reported;
        stub::fail_at = -1;
        right = t->to_host(dst.data(), src.data(), src.size(), nullptr) == hipSuccess && dst == src && right;
    }
    std::printf("%d %.3f %d %d\n", threads(), first, (int)right, (int)reported);
}
