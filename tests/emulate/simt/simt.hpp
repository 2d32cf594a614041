// simt.hpp — one wave on the CPU: 64 fibers that run until an operation across lanes, which
// is carried out once all of them have come to it.  Lanes that come to different operations, or
// that end while others wait, stop the program: such code is not wave-uniform.
#pragma once
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <memory>
#include <vector>

// Saves the callee-saved registers and the stack pointer in *from, and goes on at `to`.
extern "C" void simt_switch(void **from, void *to);
__asm__(
    ".text\n.globl simt_switch\nsimt_switch:\n"
    "pushq %rbp\npushq %rbx\npushq %r12\npushq %r13\npushq %r14\npushq %r15\n"
    "movq %rsp, (%rdi)\nmovq %rsi, %rsp\n"
    "popq %r15\npopq %r14\npopq %r13\npopq %r12\npopq %rbx\npopq %rbp\nret\n");

namespace simt {

struct Index {
    unsigned x, y;
};
enum class Op { kNone, kBallot, kReadLane, kBarrier, kEnd };

struct Fiber {
    void *sp = nullptr;
    Op op = Op::kNone;
    uint64_t value = 0, result = 0;
    int argument = 0;
    std::unique_ptr<char[]> stack;
};

constexpr size_t kStack = 256 << 10;
inline Fiber g_fibers[64];
inline void *g_main = nullptr;
inline int g_lane = 0;
inline const std::function<void()> *g_body = nullptr;
inline uint64_t g_operations = 0;  // operations across lanes since the start

inline int lane() { return g_lane; }

inline void entry() {
    (*g_body)();
    g_fibers[g_lane].op = Op::kEnd;
    simt_switch(&g_fibers[g_lane].sp, g_main);
    abort();
}

inline uint64_t wait(Op op, uint64_t value, int argument = 0) {
    Fiber &f = g_fibers[g_lane];
    f.op = op;
    f.value = value;
    f.argument = argument;
    simt_switch(&f.sp, g_main);
    return f.result;
}
inline uint64_t ballot(bool p) { return wait(Op::kBallot, p); }
inline uint64_t read_lane(uint64_t v, int from) { return wait(Op::kReadLane, v, from); }
inline void barrier() { wait(Op::kBarrier, 0); }

inline int frexp_exp(double v) {
    int e = 0;
    (void)std::frexp(v, &e);
    return e;
}
inline double frexp_mant(double v) {
    int e = 0;
    return std::frexp(v, &e);
}

// Runs `body` in all 64 lanes.
inline void run(const std::function<void()> &body) {
    g_body = &body;
    for (Fiber &f : g_fibers) {
        if (!f.stack) f.stack.reset(new char[kStack]);
        void **top = (void **)(((uintptr_t)f.stack.get() + kStack) & ~(uintptr_t)15);
        *--top = nullptr;            // the stack as at a function's first instruction
        *--top = (void *)&entry;     // simt_switch returns here
        for (int k = 0; k < 6; ++k) *--top = nullptr;
        f.sp = top;
    }
    for (;;) {
        for (g_lane = 0; g_lane < 64; ++g_lane) simt_switch(&g_main, g_fibers[g_lane].sp);
        const Op op = g_fibers[0].op;
        uint64_t mask = 0;
        for (int l = 0; l < 64; ++l) {
            const Fiber &f = g_fibers[l];
            if (f.op != op || (op == Op::kReadLane && f.argument != g_fibers[0].argument)) {
                fprintf(stderr, "lanes 0 and %d part\n", l);
                exit(3);
            }
            mask |= (f.value & 1) << l;
        }
        if (op == Op::kEnd) return;
        ++g_operations;
        const uint64_t result = op == Op::kReadLane ? g_fibers[g_fibers[0].argument].value : mask;
        for (Fiber &f : g_fibers) f.result = result;
    }
}

}  // namespace simt
