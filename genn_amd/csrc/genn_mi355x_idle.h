// Part of libgenn_mi355x.so: included by genn_mi355x.hip only (one translation unit).
//
// The thread that gives memory back which the library has kept long enough (freed device blocks, genn_mi355x_pool.h; freed pinned
// host memory, genn_mi355x_transfer.h).  It is started when memory is first kept, sleeps until something is due and ends
// with the process, before the HIP runtime does.  Where it cannot be started, kept memory goes back when memory is next asked for or freed.
#ifndef GENN_MI355X_IDLE_H
#define GENN_MI355X_IDLE_H

#include <condition_variable>
#include <thread>
#include <unistd.h>

namespace
{
using IdleClock = std::chrono::steady_clock;
using IdleTime = IdleClock::time_point;

// until when memory freed now is kept (times as long as device memory is)
IdleTime idleUntil(double times = 1.0)
{
    const char *e = getenv("GENNMI_POOL_SECONDS");
    const double seconds = times * (e ? std::min(1e6, std::max(0.0, atof(e))) : 10.0);
    return IdleClock::now() + std::chrono::duration_cast<IdleClock::duration>(std::chrono::duration<double>(seconds));
}

// Give back what is due; when the next is (IdleTime::max(): nothing is kept)
IdleTime poolReleaseOld();
IdleTime pinnedReleaseOld();

struct IdleThread
{
    std::mutex mutex;
    std::condition_variable changed;
    IdleTime due = IdleTime::max();
    bool started = false, stop = false;
    pid_t process = 0;
    std::thread thread;
};
IdleThread &idleThread()
{
    static IdleThread *t = new IdleThread;      // (never destroyed: the process may end without its exit handlers)
    return *t;
}

void idleLoop()
{
    IdleThread &t = idleThread();
    // (a stream that some other thread is capturing is none of this thread's business)
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    std::unique_lock<std::mutex> lock(t.mutex);
    while(!t.stop) {
        if(t.due == IdleTime::max()) { t.changed.wait(lock); continue; }
        if(IdleClock::now() < t.due) { t.changed.wait_until(lock, IdleTime(t.due)); continue; }
        t.due = IdleTime::max();
        lock.unlock();
        const IdleTime next = std::min(poolReleaseOld(), pinnedReleaseOld());
        lock.lock();
        t.due = std::min(t.due, next);
    }
}

// The thread looks at what is kept at this time, if not before.
void releaseIdleAt(IdleTime when)
{
    IdleThread &t = idleThread();
    std::lock_guard<std::mutex> lock(t.mutex);
    if(t.stop || when >= t.due) { return; }
    t.due = when;
    if(t.started) { t.changed.notify_one(); return; }
    try { t.thread = std::thread(idleLoop); }
    catch(const std::exception&) { t.due = IdleTime::max(); return; }
    t.started = true;
    t.process = getpid();
    // (registered after the runtime's own handlers, and so run before them)
    std::atexit([] {
        IdleThread &t = idleThread();
        if(getpid() != t.process) { return; }       // (a forked child has no such thread)
        { std::lock_guard<std::mutex> lock(t.mutex); t.stop = true; }
        t.changed.notify_one();
        t.thread.join();
    });
}
}   // namespace

#endif
