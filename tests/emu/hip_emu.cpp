// Workgroup execution for the host emulation (see hip_emu.hpp).
#include "hip_emu.hpp"

#include <ucontext.h>

#include <memory>
#include <mutex>
#include <vector>

#ifdef __SANITIZE_ADDRESS__
#include <sanitizer/common_interface_defs.h>
#endif

namespace gms_emu {

thread_local gms_emu_dim3 thread_idx = {0, 0, 0};
gms_emu_dim3 block_idx = {0, 0, 0}, block_dim = {1, 1, 1}, grid_dim = {1, 1, 1};

namespace {
// The threads of a workgroup are fibers of the launching host thread.  A
// fiber runs until it meets a wave or workgroup barrier; the scheduler in
// launch() lets it go on when every live fiber of its wave (workgroup) waits
// at one.  (One host thread per GPU thread spent nearly all its time in
// futex calls.)  Fibers run one after another, so a missing barrier shows only
// when the reader runs before the writer: every other workgroup runs its waves
// and lanes in descending order, and the next launch the others.  A race that
// needs two fibers between the same barriers to interleave does not show.
enum class State { ready, at_wave, at_block, done };
constexpr size_t kStack = 96 * 1024;
struct Fiber {
    ucontext_t ctx;
    std::unique_ptr<char[]> stack;
    State state = State::done;
    void* fake = nullptr;
};
std::vector<std::unique_ptr<Fiber>> g_fibers;
ucontext_t g_sched;
void* g_sched_fake = nullptr;
const void* g_sched_bottom = nullptr;
size_t g_sched_size = 0;
std::function<void()>* g_body = nullptr;
uint32_t g_current = 0;
uint32_t g_wave_buf[1024];
std::mutex g_launch_mutex;

#ifdef __SANITIZE_ADDRESS__
void leave(void** fake, const void* bottom, size_t size) {
    __sanitizer_start_switch_fiber(fake, bottom, size);
}
void arrive(void* fake, const void** bottom, size_t* size) {
    __sanitizer_finish_switch_fiber(fake, bottom, size);
}
#else
void leave(void**, const void*, size_t) {}
void arrive(void*, const void**, size_t*) {}
#endif

void fiber_main() {
    arrive(nullptr, &g_sched_bottom, &g_sched_size);
    (*g_body)();
    Fiber& f = *g_fibers[g_current];
    f.state = State::done;
    leave(nullptr, g_sched_bottom, g_sched_size);  // never comes back
    swapcontext(&f.ctx, &g_sched);
}

void run_fiber(uint32_t i) {
    Fiber& f = *g_fibers[i];
    g_current = i;
    thread_idx = {i, 0, 0};
    leave(&g_sched_fake, f.stack.get(), kStack);
    swapcontext(&g_sched, &f.ctx);
    arrive(g_sched_fake, nullptr, nullptr);
}

void wait_at(State s) {
    Fiber& f = *g_fibers[g_current];
    f.state = s;
    leave(&f.fake, g_sched_bottom, g_sched_size);
    swapcontext(&f.ctx, &g_sched);
    arrive(f.fake, &g_sched_bottom, &g_sched_size);
}
}  // namespace

void syncthreads() { wait_at(State::at_block); }

struct WaveBarrier {
    void arrive_and_wait() { wait_at(State::at_wave); }
};
static WaveBarrier wave_barrier() { return {}; }

uint32_t update_dpp(uint32_t old, uint32_t src, int ctrl, int row_mask, int bank_mask,
                    bool bound_ctrl) {
    const uint32_t lane = thread_idx.x & 63u, wave_base = thread_idx.x & ~63u;
    uint32_t* buf = g_wave_buf + wave_base;
    buf[lane] = src;
    wave_barrier().arrive_and_wait();
    const int row = (int)(lane >> 4), bank = (int)((lane >> 2) & 3u);
    uint32_t r;
    if (!((row_mask >> row) & 1) || !((bank_mask >> bank) & 1)) {
        r = old;  // lane not written
    } else {
        int s = -1;
        if (ctrl >= 0x111 && ctrl <= 0x11F) {  // row_shr:n
            const int sh = ctrl - 0x110;
            if ((int)(lane & 15u) >= sh) s = (int)lane - sh;
        } else if (ctrl == 0x142) {  // row_bcast:15
            if (row >= 1) s = row * 16 - 1;
        } else if (ctrl == 0x143) {  // row_bcast:31
            if (row >= 2) s = 31;
        } else {
            fprintf(stderr, "hip_emu: unsupported dpp control 0x%x\n", ctrl);
            abort();
        }
        r = s >= 0 ? buf[s] : (bound_ctrl ? 0u : old);
    }
    wave_barrier().arrive_and_wait();
    return r;
}

void wave_sync() { wave_barrier().arrive_and_wait(); }

int readlane(int x, int lane) {
    const uint32_t wave_base = thread_idx.x & ~63u;
    uint32_t* buf = g_wave_buf + wave_base;
    buf[thread_idx.x & 63u] = (uint32_t)x;
    wave_barrier().arrive_and_wait();
    const int r = (int)buf[lane & 63];
    wave_barrier().arrive_and_wait();
    return r;
}

uint64_t ballot(bool pred) {
    const uint32_t wave_base = thread_idx.x & ~63u;
    uint32_t* buf = g_wave_buf + wave_base;
    buf[thread_idx.x & 63u] = pred ? 1u : 0u;
    wave_barrier().arrive_and_wait();
    uint64_t m = 0;
    const uint32_t lanes = block_dim.x - wave_base < 64u ? block_dim.x - wave_base : 64u;
    for (uint32_t l = 0; l < lanes; ++l) m |= (uint64_t)(buf[l] & 1u) << l;
    wave_barrier().arrive_and_wait();
    return m;
}

void launch(dim3 grid, dim3 block, std::function<void()> body) {
    std::lock_guard<std::mutex> lk(g_launch_mutex);
    const uint32_t nt = block.x;
    if (nt == 0 || nt > 1024 || (nt % 64 != 0 && nt > 64)) {
        fprintf(stderr, "hip_emu: unsupported block size %u\n", nt);
        abort();
    }
    grid_dim = {grid.x, 1, 1};
    block_dim = {nt, 1, 1};
    while (g_fibers.size() < nt) {
        g_fibers.push_back(std::make_unique<Fiber>());
        g_fibers.back()->stack.reset(new char[kStack]);
    }
    g_body = &body;
    static uint32_t launches = 0;
    ++launches;
    const uint32_t waves = (nt + 63) / 64;
    for (uint32_t b = 0; b < grid.x; ++b) {
        const bool down = ((b + launches) & 1u) != 0;
        block_idx = {b, 0, 0};
        for (uint32_t t = 0; t < nt; ++t) {
            Fiber& f = *g_fibers[t];
            getcontext(&f.ctx);
            f.ctx.uc_stack.ss_sp = f.stack.get();
            f.ctx.uc_stack.ss_size = kStack;
            f.ctx.uc_link = nullptr;
            makecontext(&f.ctx, fiber_main, 0);
            f.state = State::ready;
        }
        for (bool live = true; live;) {
            live = false;
            for (uint32_t v = 0; v < waves; ++v) {  // every wave up to its workgroup barrier
                const uint32_t w = (down ? waves - 1 - v : v) * 64;
                const uint32_t end = w + 64 < nt ? w + 64 : nt;
                for (bool again = true; again;) {
                    uint32_t at_wave = 0, at_block = 0;
                    for (uint32_t i = w; i < end; ++i) {
                        const uint32_t t = down ? w + end - 1 - i : i;
                        if (g_fibers[t]->state == State::ready) run_fiber(t);
                        at_wave += g_fibers[t]->state == State::at_wave;
                        at_block += g_fibers[t]->state == State::at_block;
                    }
                    if (at_wave && at_block) {
                        fprintf(stderr, "hip_emu: a wave waits at two different barriers\n");
                        abort();
                    }
                    again = at_wave != 0;
                    live = live || at_block != 0;
                    for (uint32_t t = w; t < end && again; ++t)
                        if (g_fibers[t]->state == State::at_wave) g_fibers[t]->state = State::ready;
                }
            }
            for (uint32_t t = 0; t < nt; ++t)
                if (g_fibers[t]->state == State::at_block) g_fibers[t]->state = State::ready;
        }
    }
    thread_idx = {0, 0, 0};
}

std::atomic<uint64_t> alloc_calls{0};
std::atomic<uint32_t> refuse_pinned{0};
thread_local int last_error = 0;
}  // namespace gms_emu

// Allocation calls (hipMalloc, hipFree, hipHostMalloc, hipHostFree) so far.
extern "C" uint64_t gms_emu_alloc_calls() { return gms_emu::alloc_calls.load(); }

// The next `count` pinned allocations fail.
extern "C" void gms_emu_refuse_pinned(uint32_t count) { gms_emu::refuse_pinned = count; }
