// Host program for the test of the order of resident time loops (myea_amd/csrc/myea_loop_order.h): a stand-in for the device counts the loops
// that were launched, that run, and that run beside each other.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <thread>

#include "../../myea_amd/csrc/myea_loop_order.h"

namespace {

constexpr int kStreams = 4;
std::atomic<int> g_running[kStreams], g_idle_waits, g_awaits;
std::atomic<int> g_mark{-1};   // the stream whose loop the mark is behind
std::atomic<bool> g_capturing[kStreams];

struct Device {
    using Stream = int;
    bool capturing(Stream s) { return g_capturing[s]; }
    void await(Stream) { ++g_awaits; if (g_mark >= 0) g_running[g_mark] = 0; }
    bool mark(Stream s) { g_mark = s; return true; }
    void wait_idle() { ++g_idle_waits; for (auto &r : g_running) r = 0; }
};
using Order = myea::LoopOrder<Device>;
using Turn = myea::LoopTurn<Device>;

int fail(const char *what) { std::printf("FAILED: %s\n", what); return 1; }
void pause() { std::this_thread::sleep_for(std::chrono::milliseconds(100)); }
bool others_run(int s)
{
    for (int o = 0; o < kStreams; ++o) if (o != s && g_running[o] > 0) return true;
    return false;
}

// the first network is between its look at the order and its launch when a second one joins and launches
int join_meanwhile()
{
    Order order;
    order.join();
    std::atomic<bool> beside{false};
    std::thread second;
    {
        Turn turn(&order, "a", 0);
        second = std::thread([&] {
            order.join();
            Turn other(&order, "b", 1);
            beside = others_run(1);
            g_running[1] = 1;
        });
        pause();
        if (others_run(0)) beside = true;
        g_running[0] = 1;
    }
    second.join();
    return beside ? fail("a network that joined meanwhile launched beside the first one's loop") : 0;
}

// a network leaves while its loop runs; another launches then
int leave_running(int networks)
{
    Order order;
    for (int i = 0; i < networks; ++i) order.join();
    {
        Turn turn(&order, "a", 0);
        g_running[0] = 1;
    }
    order.leave("a");
    if (networks == 1) order.join();
    Turn turn(&order, "b", 1);
    return others_run(1) ? fail("a loop was launched beside the one of a network that has left") : 0;
}

// ordinary turns: each loop waits for the one before it on another network's stream, not for its own; a capturing stream is left alone
int turns()
{
    Order order;
    order.join(); order.join();
    const int start = g_awaits;
    for (int i = 0; i < 3; ++i)
        for (int s = 0; s < 2; ++s) {
            for (int twice = 0; twice < 2; ++twice) {
                Turn turn(&order, s ? "b" : "a", s);
                if (others_run(s)) return fail("two loops beside each other");
                g_running[s] = 1;
            }
        }
    if (g_awaits - start != 5) return fail("a network waits for the other's loop, and only for that");
    g_capturing[2] = true;
    { Turn turn(&order, "c", 2); }
    g_capturing[2] = false;
    if (g_awaits - start != 5 || g_mark != 1) return fail("a capturing stream is left alone");
    { Turn none(nullptr, "a", 0); }
    return 0;
}

}  // namespace

int main(int argc, char **argv)
{
    const char *what = argc > 1 ? argv[1] : "";
    if (!std::strcmp(what, "join")) return join_meanwhile();
    if (!std::strcmp(what, "leave-one")) return leave_running(1);
    if (!std::strcmp(what, "leave-two")) return leave_running(2);
    if (!std::strcmp(what, "leave-three")) return leave_running(3);
    if (!std::strcmp(what, "turns")) return turns();
    return fail("usage: loop_order_check join | leave-one | leave-two | leave-three | turns");
}
