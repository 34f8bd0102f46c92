// Counts what the queue of a rank's waiting calls (host/call_queue.h) moves and holds.  argv: calls that wait at the start,
// then that many are taken, one more being added after every second one.  Prints moves of a call behind its way in and out, the
// largest capacity, the capacity at the end, calls out of order.
#include <cstdio>
#include <cstdlib>

#include "host/call_queue.h"

static unsigned long long g_moves = 0;

struct Call {
    long number = -1;
    explicit Call(long n) : number(n) {}
    Call(Call &&o) noexcept : number(o.number) { ++g_moves; }
    Call &operator=(Call &&o) noexcept
    {
        number = o.number;
        ++g_moves;
        return *this;
    }
};

int main(int, char **argv)
{
    const long waiting = std::atol(argv[1]);
    ops_hccl::CallQueue<Call> q;
    long in = 0;
    for (; in < waiting; ++in) q.Push(Call(in));
    g_moves = 0;
    size_t most = q.capacity();
    long out = 0;
    long wrong = 0;
    while (!q.empty()) {
        wrong += q.Take().number != out++;
        if (out % 2 == 0 && out < waiting) q.Push(Call(in++));
        if (q.capacity() > most) most = q.capacity();
    }
    std::printf("%llu %zu %zu %ld %ld\n", g_moves, most, q.capacity(), wrong, out);
    return 0;
}
