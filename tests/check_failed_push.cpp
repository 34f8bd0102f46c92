// A rank's call for which there is no memory left leaves the world as it was: it does not count as waiting, and the collective
// runs once the rank has called again.  Dry world; prints the number of collectives that ran.
#include <cstdio>
#include <cstdlib>
#include <new>

#include "hccl.h"
#include "hccl_comm.h"
#include "hcclx.h"

static bool g_fail = false;

void *operator new(size_t n)
{
    if (g_fail) throw std::bad_alloc();
    if (void *p = std::malloc(n != 0 ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

int main()
{
    HcclComm comm[2] = {nullptr, nullptr};
    if (hcclxCommInitAll(2, 8u << 20, 1, comm) != HCCL_SUCCESS) return 2;
    char *const at = reinterpret_cast<char *>(1ull << 30);
    auto reduce = [&](int r) {
        return HcclAllReduce(at + (r << 20), at + ((r + 8) << 20), 100, HCCL_DATA_TYPE_FP32, HCCL_REDUCE_SUM, comm[r], at);
    };
    auto ran = [&] {
        hcclxLastOpInfo info = {};
        return hcclxCommGetLastOpInfo(comm[0], &info) == HCCL_SUCCESS && info.algName[0] != 0;
    };
    bool refused = false;
    g_fail = true;
    try {
        (void)reduce(0);
    } catch (const std::bad_alloc &) {
        refused = true;
    }
    g_fail = false;
    if (!refused) return 3;
    if (reduce(1) != HCCL_SUCCESS || ran()) return 4;   // it waits for rank 0
    if (reduce(0) != HCCL_SUCCESS || !ran()) return 5;
    std::printf("ok\n");
    return 0;
}
