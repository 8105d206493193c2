// myea_loop_order.h — the order of the resident time loops of a process's networks on a device (host; the device is a template argument,
// so that the order can be tested without one).
//
// Two resident loops at once may each hold compute units that the other's workgroups wait for.  So while more than one network of the
// process has such layers on a device, a loop waits (on the device) for the loop launched before it on another network's stream; a
// stream that is being captured is left alone.  The lock is held from the look at the number of networks until the loop is launched, so that
// one that joins meanwhile finds it; one that leaves waits for its loops before the others forget it.
#pragma once

#include <mutex>

namespace myea {

// Device: Stream; capturing(stream); await(stream), which has the stream wait for the mark; mark(stream), which sets the mark behind what the
// stream holds (false: it could not); wait_idle()
template <class Device>
struct LoopOrder {
    std::mutex mutex;
    int networks = 0;
    const void *owner = nullptr;   // the network whose loop the mark is behind
    Device device;

    void join()
    {
        std::lock_guard<std::mutex> lock(mutex);
        if (++networks == 2) device.wait_idle();   // the first network's loops so far have left no mark behind
    }
    void leave(const void *net)
    {
        std::lock_guard<std::mutex> lock(mutex);
        device.wait_idle();
        --networks;
        if (owner == net) owner = nullptr;
    }
};

// held while a loop is launched
template <class Device>
struct LoopTurn {
    LoopOrder<Device> *const order;
    const void *const net;
    const typename Device::Stream stream;
    bool marks = false;

    LoopTurn(LoopOrder<Device> *o, const void *n, typename Device::Stream s) : order(o), net(n), stream(s)
    {
        if (!order) return;
        order->mutex.lock();
        marks = order->networks >= 2 && !order->device.capturing(stream);
        if (marks && order->owner && order->owner != net) order->device.await(stream);
    }
    ~LoopTurn()
    {
        if (!order) return;
        if (marks && order->device.mark(stream)) order->owner = net;
        order->mutex.unlock();
    }
    LoopTurn(const LoopTurn &) = delete;
    LoopTurn &operator=(const LoopTurn &) = delete;
};

}  // namespace myea
