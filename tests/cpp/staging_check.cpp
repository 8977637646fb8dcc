// Drives lbm_amd/csrc/staging.h over a host stand-in of the runtime
// (host_hip/hip/hip_runtime.h) for tests/test_staging.py:
//   staging_check copy out|in BYTES [BYTES ...]   the pieces of one call, twice
//   staging_check odd out|in BYTES                device memory at an odd address
//   staging_check pinned out|in BYTES             pinned caller memory
//   staging_check nothread out|in BYTES N         the N-th thread cannot be made
//   staging_check error out|in BYTES N            the N-th chunk's launch fails
// Prints "ok", whether chunks were made, and the runtime's copies and the launches; any wrong byte ends it with status 1.
#include <cstdio>
#include <cstdlib>
#include <new>
#include <string>

#include "../../lbm_amd/csrc/staging.h"

// the N-th allocation from now on in this thread fails (a thread's state is one
// allocation in the thread that makes it)
static thread_local int fail_new = -1;
void *operator new(size_t n) {
    if (fail_new >= 0 && fail_new-- == 0) throw std::bad_alloc();
    if (void *p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

static FakeStream s;  // the object's stream

// a byte for each place, without the period of a chunk
static char byte_at(size_t b, unsigned seed) {
    const uint64_t z = (b + ((uint64_t)seed << 40)) * 0x9E3779B97F4A7C15ull;
    return (char)((z ^ (z >> 29)) * 0xBF58476D1CE4E5B9ull >> 56);
}

static bool fill_and_compare(Staging &st, bool out, const std::vector<size_t> &sizes, bool pinned, unsigned seed,
                             hipError_t expect, size_t shift = 0) {
    constexpr size_t kGuard = 64;
    std::vector<std::vector<char>> dev(sizes.size()), ref(sizes.size());
    std::vector<char *> host(sizes.size());
    std::vector<Piece> pieces;
    for (size_t i = 0; i < sizes.size(); ++i) {
        const size_t n = sizes[i] + 2 * kGuard + shift;
        if (pinned) (void)hipHostMalloc((void **)&host[i], n, hipHostMallocDefault);
        else host[i] = (char *)std::malloc(n);
        dev[i].assign(n, 'd');  // (device memory from dev + shift on)
        std::memset(host[i], 'h', n);
        ref[i].resize(sizes[i]);
        for (size_t b = 0; b < sizes[i]; ++b) ref[i][b] = byte_at(b, 97 * seed + (unsigned)i);
        char *const from = out ? dev[i].data() + shift : host[i];
        std::memcpy(from + kGuard, ref[i].data(), sizes[i]);
        pieces.push_back({host[i] + kGuard, dev[i].data() + shift + kGuard, sizes[i]});
    }
    const hipError_t e = st.copy(3, &s, pieces.data(), (int)pieces.size(), out);
    if (e == hipSuccess && !out) (void)hipStreamSynchronize(&s);
    bool ok = e == expect;
    if (e == hipSuccess)
        for (size_t i = 0; i < sizes.size(); ++i) {
            const char *to = out ? host[i] : dev[i].data() + shift;
            const char mark = out ? 'h' : 'd';
            ok = ok && std::memcmp(to + kGuard, ref[i].data(), sizes[i]) == 0;
            for (size_t b = 0; b < kGuard; ++b) ok = ok && to[b] == mark && to[kGuard + sizes[i] + b] == mark;
        }
    for (char *h : host) {
        if (pinned) (void)hipHostFree(h);
        else std::free(h);
    }
    return ok;
}

int main(int argc, char **argv) {
    if (argc < 4) return 2;
    const std::string cmd = argv[1];
    const bool out = std::string(argv[2]) == "out";
    std::vector<size_t> sizes{std::strtoull(argv[3], nullptr, 10)};
    Staging st;
    bool ok = true;
    if (cmd == "copy") {
        for (int i = 4; i < argc; ++i) sizes.push_back(std::strtoull(argv[i], nullptr, 10));
        for (unsigned seed = 1; seed <= 2; ++seed)  // the second call meets the first one's chunks
            ok = ok && fill_and_compare(st, out, sizes, false, seed, hipSuccess);
    } else if (cmd == "odd") {
        ok = fill_and_compare(st, out, sizes, false, 1, hipSuccess, 1);
    } else if (cmd == "pinned") {
        ok = fill_and_compare(st, out, sizes, true, 1, hipSuccess);
        --fake().host_mallocs;  // the caller's own
    } else if (cmd == "nothread" && argc == 5) {
        ok = fill_and_compare(st, out, sizes, false, 1, hipSuccess);  // the chunks are there
        const int n = std::atoi(argv[4]);
        // (the list of chunks is the call's first allocation, the threads' states the next ones)
        std::vector<char> dev(sizes[0], 'd'), host(sizes[0], 'h');
        std::vector<char> &from = out ? dev : host, &to = out ? host : dev;
        for (size_t b = 0; b < sizes[0]; ++b) from[b] = byte_at(b, 1);
        const std::vector<char> want = from;
        const Piece p{host.data(), dev.data(), sizes[0]};
        s.ops.reserve(4096);
        fail_new = 1 + n;
        const hipError_t e = st.copy(3, &s, &p, 1, out);
        fail_new = -1;
        (void)hipStreamSynchronize(&s);
        ok = ok && e == hipSuccess && to == want;
    } else if (cmd == "error" && argc == 5) {
        fake().fail_launch = std::atoi(argv[4]);
        ok = fill_and_compare(st, out, sizes, false, 1, hipErrorUnknown);
        fake().fail_launch = -1;
        ok = ok && fill_and_compare(st, out, sizes, false, 2, hipSuccess);  // and the next call is whole
    } else {
        return 2;
    }
    const bool clean = hipGetLastError() == hipSuccess || cmd == "error";
    st.release();
    std::printf("%s chunks=%d copies=%d launches=%d\n", ok ? (clean ? "ok" : "an error is left behind") : "wrong",
                fake().host_mallocs, fake().copies, fake().launches);
    return ok && clean ? 0 : 1;
}
