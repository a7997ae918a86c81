// Runs a kernel on the CPU: an operating-system thread per workgroup, a stack per lane (x86-64).
#pragma once
#include <stddef.h>
namespace simt {
struct Launch {
    int groups, threads;         // workgroups, threads of each (a multiple of 64)
    size_t lds;                  // bytes of dynamic LDS
    unsigned seed;               // of the order in which wavefronts run
    int xccs;                    // workgroup b runs on XCC b % xccs
    void (*kernel)(const void *args);
    const void *args;
};
void run(const Launch &launch);  // returns when all workgroups have ended

// Memory whose end, up to the alignment, is followed by a page that no access survives.
class Guarded {
public:
    explicit Guarded(size_t bytes, size_t alignment);
    ~Guarded();
    Guarded(const Guarded &) = delete;
    void *get() const { return at; }
private:
    void *at, *pages;
    size_t length;
};
}
