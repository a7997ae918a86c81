// Lanes, wavefronts and workgroups for hip/hip_runtime.h.  Built without sanitizers; what ThreadSanitizer must know, it is told:
// a wavefront is one thread of execution to it (its lanes run in step on the device), barriers order wavefronts.
#include "simt.h"
#include "hip/hip_runtime.h"
#include <stdio.h>
#include <stdlib.h>
#include <sys/mman.h>
#include <memory>
#include <random>
#include <thread>
#include <vector>

extern "C" {
void *__tsan_create_fiber(unsigned) __attribute__((weak));
void *__tsan_get_current_fiber() __attribute__((weak));
void __tsan_destroy_fiber(void *) __attribute__((weak));
void __tsan_switch_to_fiber(void *, unsigned) __attribute__((weak));
void __tsan_acquire(void *) __attribute__((weak));
void __tsan_release(void *) __attribute__((weak));
void simt_switch(void **save, void *to);
}
// saves the callee-saved registers on the stack, leaves the stack pointer in *save and goes on with the stack `to`
asm(R"(.text
.globl simt_switch
.type simt_switch,@function
simt_switch:
    pushq %rbp; pushq %rbx; pushq %r12; pushq %r13; pushq %r14; pushq %r15
    movq %rsp, (%rdi)
    movq %rsi, %rsp
    popq %r15; popq %r14; popq %r13; popq %r12; popq %rbx; popq %rbp
    ret
)");

namespace simt {
thread_local Where where;
namespace {
constexpr size_t kStack = 512 * 1024;
enum State { kReady, kWaiting, kEnded };
struct Wave;
struct Lane { Where where; void *sp = nullptr; char *stack = nullptr; State state = kReady; Wave *wave = nullptr; };
struct Wave {
    Lane lanes[64];
    uint64_t values[2][64];   // (a lane can be one meeting ahead of another, not two)
    int turn = 0, arrived = 0, ready = 64;
    Kind kind = kSync;
    void *fiber = nullptr;
};
struct Group {
    const Launch *launch; int index;
    std::vector<std::unique_ptr<Wave>> waves;
    std::unique_ptr<Guarded> lds;
    void *scheduler = nullptr, *own_fiber = nullptr, *fiber = nullptr;
    Lane *now = nullptr;
    int live = 0, at_barrier = 0, phase = 0;
    Kind barrier_kind = kBarrier;
    bool all[2] = {true, true};
    char phases[2];           // what ThreadSanitizer knows the barrier by
};
thread_local Group *group;
char launched, ended;
[[noreturn]] void wrong(const char *what) { fprintf(stderr, "simt: workgroup %d, thread %d: %s\n", group->index, group->now ? group->now->where.thread.x : -1, what); abort(); }
void to_scheduler() { Lane *const l = group->now; l->where = where; simt_switch(&l->sp, group->scheduler); }
void acquire(void *p) { if (__tsan_acquire) __tsan_acquire(p); }
void release(void *p) { if (__tsan_release) __tsan_release(p); }
void enter() {
    acquire(&launched);
    group->launch->kernel(group->launch->args);
    Lane *const l = group->now;
    if (l->wave->arrived != 0) wrong("ends while others of its wavefront wait");
    release(&ended);
    l->state = kEnded; l->wave->ready--; group->live--;
    to_scheduler();
}
void run_group(const Launch &launch, int index) {
    Group g;
    group = &g;
    g.launch = &launch; g.index = index; g.live = launch.threads;
    g.lds.reset(new Guarded(launch.lds, 16));
    std::mt19937 rng(launch.seed * 1000003u + (unsigned)index);
    for (size_t i = 0; i < launch.lds; i++) static_cast<char *>(g.lds->get())[i] = (char)(rng() >> 5);   // (LDS holds anything at first)
    if (__tsan_get_current_fiber) g.own_fiber = g.fiber = __tsan_get_current_fiber();
    for (int w = 0; w < launch.threads / 64; w++) {
        g.waves.emplace_back(new Wave);
        Wave &wave = *g.waves.back();
        if (__tsan_create_fiber) wave.fiber = __tsan_create_fiber(0);
        for (int i = 0; i < 64; i++) {
            Lane &l = wave.lanes[i];
            l.wave = &wave;
            l.where = Where{{w * 64 + i, 0, 0}, {index, 0, 0}, {launch.threads, 1, 1}, i};
            l.stack = (char *)mmap(nullptr, kStack, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
            if (l.stack == MAP_FAILED) wrong("no memory for a stack");
            void **top = (void **)(l.stack + kStack - 64);
            *--top = nullptr;               // (as a call would have left it: the stack is 16 bytes off a multiple by one word)
            *--top = (void *)&enter;
            for (int k = 0; k < 6; k++) *--top = nullptr;
            l.sp = top;
        }
    }
    while (g.live > 0) {
        int ready = 0;
        for (auto &w : g.waves) ready += w->ready > 0;
        if (ready == 0) {
            for (auto &w : g.waves) fprintf(stderr, "simt: wavefront of thread %d: %d lanes at operation %d\n", w->lanes[0].where.thread.x, w->arrived, (int)w->kind);
            wrong("no lane can go on");
        }
        int k = (int)(rng() % (unsigned)ready);
        Wave *wave = nullptr;
        for (auto &w : g.waves) if (w->ready > 0 && k-- == 0) { wave = w.get(); break; }
        if (wave->fiber && g.fiber != wave->fiber) { __tsan_switch_to_fiber(wave->fiber, 1); g.fiber = wave->fiber; }
        for (Lane &l : wave->lanes) {
            if (l.state != kReady) continue;
            g.now = &l; where = l.where;
            simt_switch(&g.scheduler, l.sp);
        }
    }
    if (g.own_fiber && g.fiber != g.own_fiber) __tsan_switch_to_fiber(g.own_fiber, 1);
    acquire(&ended);
    for (auto &w : g.waves) {
        if (w->fiber) __tsan_destroy_fiber(w->fiber);
        for (Lane &l : w->lanes) munmap(l.stack, kStack);
    }
}
}  // namespace

const uint64_t *together(Kind kind, uint64_t mine) {
    Lane *const l = group->now;
    Wave *const w = l->wave;
    if (w->arrived == 0) w->kind = kind;
    else if (w->kind != kind) wrong("lanes of a wavefront meet at different operations");
    const int turn = w->turn;
    w->values[turn][where.lane] = mine;
    if (++w->arrived == 64) {
        w->arrived = 0; w->turn ^= 1;
        for (Lane &o : w->lanes) if (o.state == kWaiting) { o.state = kReady; w->ready++; }
    } else { l->state = kWaiting; w->ready--; to_scheduler(); }
    return w->values[turn];
}

bool barrier(Kind kind, bool mine) {
    Group *const g = group;
    Lane *const l = g->now;
    if (g->at_barrier == 0) g->barrier_kind = kind;
    else if (g->barrier_kind != kind) wrong("wavefronts meet at different barriers");
    const int phase = g->phase;
    release(&g->phases[phase]);
    g->all[phase] = g->all[phase] && mine;
    if (++g->at_barrier == g->launch->threads) {
        g->at_barrier = 0; g->phase ^= 1; g->all[phase ^ 1] = true;
        for (auto &w : g->waves)
            for (Lane &o : w->lanes) if (o.state == kWaiting) { o.state = kReady; w->ready++; }
    } else { l->state = kWaiting; l->wave->ready--; to_scheduler(); }
    acquire(&g->phases[phase]);
    return g->all[phase];
}

void pause() {
    static thread_local unsigned count;
    if ((++count & 255u) == 0) std::this_thread::yield();
    to_scheduler();
}

void *dynamic_lds() { return group->lds->get(); }
int xcc() { return group->index % group->launch->xccs; }

Guarded::Guarded(size_t bytes, size_t alignment) {
    const size_t page = 4096, held = (bytes + page - 1) / page * page;
    length = held + 2 * page;
    pages = mmap(nullptr, length, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
    if (pages == MAP_FAILED || (held && mprotect((char *)pages + page, held, PROT_READ | PROT_WRITE) != 0)) { fprintf(stderr, "simt: no memory\n"); abort(); }
    at = (char *)pages + page + (held - bytes) / alignment * alignment;
}
Guarded::~Guarded() { munmap(pages, length); }

void run(const Launch &launch) {
    release(&launched);
    std::vector<std::thread> threads;
    for (int b = 0; b < launch.groups; b++) threads.emplace_back(run_group, std::cref(launch), b);
    for (auto &t : threads) t.join();
    acquire(&ended);
}
}  // namespace simt
