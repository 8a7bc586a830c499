// Runs k_bin_direct (kernel.inc, cut from the library's source) for one bin on
// the CPU: boxes-file n bins-a-row bin up|down; prints the bin's triangles.
// A fiber a thread.  A wave's fibers meet at every ballot; a wave runs until
// all its fibers stand at a barrier before the next wave runs, in ascending or
// descending order.  Exit code 3: the waves stand at different barriers.
#include <ucontext.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

using std::min;
struct uint2 { uint32_t x, y; };
static uint2 make_uint2(uint32_t x, uint32_t y) { return uint2{x, y}; }
struct Dim { uint32_t x; };
static Dim threadIdx, blockIdx;

struct DirectParams {
    const uint2* boxes;
    uint32_t n, nbx, stride;
    uint32_t *list, *start, *end;
    int masks;
};
static uint32_t direct_mask(const DirectParams&, uint32_t t, uint32_t, uint32_t) { return 1u << t % 16u; }
static void atomicOr(uint32_t* p, uint32_t v) { *p |= v; }
constexpr uint32_t END_MASKED = 1u << 31, MASK_ITEMS = 16;

constexpr uint32_t THREADS = 512, WAVES = THREADS / 64;
enum At { RUNS, BALLOT, BARRIER, DONE };
struct Fiber {
    ucontext_t c;
    At at = RUNS;
    int line = 0;
    bool vote = false;
    uint64_t ballot = 0;
};
static Fiber fibers[THREADS];
static ucontext_t scheduler;
static uint32_t current;

static void stop(At at, int line) {
    Fiber& f = fibers[current];
    f.at = at;
    f.line = line;
    swapcontext(&f.c, &scheduler);
}
static uint64_t ballot(bool p, int line) {
    fibers[current].vote = p;
    stop(BALLOT, line);
    return fibers[current].ballot;
}
static uint32_t count_below(uint64_t mask, uint32_t c) {
    const uint32_t lane = threadIdx.x & 63u;
    return c + (uint32_t)__builtin_popcountll(mask & ((1ull << lane) - 1));
}

#define __global__ static
#define __launch_bounds__(n)
#define __shared__ static
#define __syncthreads() stop(BARRIER, __LINE__)
#define __ballot(p) ballot(p, __LINE__)
#define __popcll(m) __builtin_popcountll(m)
#define __builtin_amdgcn_readfirstlane(v) (v)
#define __builtin_amdgcn_mbcnt_lo(m, c) count_below((uint64_t)(m), c)
#define __builtin_amdgcn_mbcnt_hi(m, c) count_below((uint64_t)(m) << 32, c)
#include "kernel.inc"
static_assert(DIRECT_THREADS == THREADS, "a fiber a thread");

static DirectParams params;
static void body() {
    k_bin_direct(params);
    stop(DONE, 0);
}

static int fail(const char* what) {
    fprintf(stderr, "%s\n", what);
    return 3;
}

int main(int argc, char** argv) {
    if (argc != 6) return 2;
    const uint32_t n = (uint32_t)atoi(argv[2]);
    std::vector<uint2> boxes(n);
    FILE* f = fopen(argv[1], "rb");
    if (!f || fread(boxes.data(), sizeof(uint2), n, f) != n) return 2;
    fclose(f);
    const uint32_t nbx = (uint32_t)atoi(argv[3]), bin = (uint32_t)atoi(argv[4]);
    const bool down = !strcmp(argv[5], "down");
    std::vector<uint32_t> list((size_t)n * (bin + 1)), start(bin + 1), end(bin + 1);
    params = DirectParams{boxes.data(), n, nbx, n, list.data(), start.data(), end.data(), down};
    blockIdx.x = bin;
    constexpr size_t STACK = 32768;
    std::vector<char> stacks(STACK * THREADS);
    for (uint32_t t = 0; t < THREADS; t++) {
        getcontext(&fibers[t].c);
        fibers[t].c.uc_stack.ss_sp = stacks.data() + STACK * t;
        fibers[t].c.uc_stack.ss_size = STACK;
        makecontext(&fibers[t].c, body, 0);
    }
    for (;;) {
        for (uint32_t k = 0; k < WAVES; k++) {
            const uint32_t w0 = 64u * (down ? WAVES - 1 - k : k);
            for (;;) {
                for (uint32_t t = w0; t < w0 + 64; t++) {
                    if (fibers[t].at != RUNS) continue;
                    current = t;
                    threadIdx.x = t;
                    swapcontext(&scheduler, &fibers[t].c);
                }
                for (uint32_t t = w0; t < w0 + 64; t++)
                    if (fibers[t].at != fibers[w0].at || fibers[t].line != fibers[w0].line)
                        return fail("the lanes of a wave are apart");
                if (fibers[w0].at != BALLOT) break;
                uint64_t m = 0;
                for (uint32_t l = 0; l < 64; l++) m |= (uint64_t)fibers[w0 + l].vote << l;
                for (uint32_t t = w0; t < w0 + 64; t++) {
                    fibers[t].ballot = m;
                    fibers[t].at = RUNS;
                }
            }
        }
        for (uint32_t t = 0; t < THREADS; t++)
            if (fibers[t].at != fibers[0].at || fibers[t].line != fibers[0].line)
                return fail("waves stand at different barriers");
        if (fibers[0].at == DONE) break;
        for (Fiber& x : fibers) x.at = RUNS;
    }
    const bool masked = end[bin] & END_MASKED;
    const uint32_t stop = masked ? start[bin] + (end[bin] >> 16 & 0x7FFFu) : end[bin];
    if (masked != (params.masks && stop - start[bin] <= MASK_ITEMS)) return fail("the form of the end");
    uint32_t all = 0;
    for (uint32_t i = start[bin]; i < stop; i++) {
        const uint32_t t = list[i] >> 16;
        if ((list[i] & 0xFFFFu) != 1u << t % 16u) return fail("an item's mask");
        all |= list[i] & 0xFFFFu;
        printf("%u\n", t);
    }
    if (masked && (end[bin] & 0xFFFFu) != all) return fail("the bin's mask");
    return 0;
}
