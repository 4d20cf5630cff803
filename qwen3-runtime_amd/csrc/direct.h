// Direct loads from global memory to LDS, and the waits that go with them. The compiler does not count
// such a load's arrival before a read of the same LDS: every wait is the program's own.
#pragma once

#define QRT_WAIT_LOADS(n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n) : "memory")
#define QRT_WAIT_LDS() asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory")
// A barrier without the fence of __syncthreads(), which would wait for every direct load to LDS
// in flight: what has to have landed is waited for by hand before it.
#define QRT_BARRIER() asm volatile("s_barrier" ::: "memory")
typedef const void __attribute__((address_space(1)))* global_ptr_t;
typedef void __attribute__((address_space(3)))* lds_ptr_t;
