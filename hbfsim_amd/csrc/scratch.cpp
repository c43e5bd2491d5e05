// scratch.cpp -- the per-device pool behind scratch.hpp.
#include "scratch.hpp"

#include <algorithm>
#include <initializer_list>
#include <mutex>
#include <new>
#include <vector>

namespace hbfamd {
namespace {

struct Block {
    void* ptr;
    std::size_t bytes;
    int device;
    bool busy;
};

std::mutex g_mu;
// never destroyed: engines may outlive this file's static objects
std::vector<Block>& g_blocks = *new std::vector<Block>;

std::size_t g_holders = 0;

// An idle block serves requests of at least half its size: a small request must not keep a large
// block from the next large one.
constexpr std::size_t kFitMost = 2;

// Takes the idle blocks of `device` (-1: of every device) out of the list, oldest first, until at
// most `keep` idle bytes remain; the caller frees them without the lock.  A block of more than
// `keep` could not stay whatever else went, so it goes before any other.
std::vector<void*> take_idle(int device, std::size_t keep)
{
    std::size_t idle = 0;
    const auto mine = [&](const Block& b) {
        return !b.busy && (device < 0 || b.device == device);
    };
    for (const Block& b : g_blocks) {
        idle += mine(b) ? b.bytes : 0;
    }
    std::vector<void*> out;
    out.reserve(g_blocks.size());  // before any block leaves the list: nothing below throws
    for (const bool large : {true, false}) {
        for (std::size_t k = 0; k < g_blocks.size() && idle > keep;) {
            if (mine(g_blocks[k]) && (!large || g_blocks[k].bytes > keep)) {
                out.push_back(g_blocks[k].ptr);
                idle -= g_blocks[k].bytes;
                g_blocks.erase(g_blocks.begin() + static_cast<std::ptrdiff_t>(k));
            } else {
                ++k;
            }
        }
    }
    return out;
}

}  // namespace

void* scratch_take(std::size_t bytes)
{
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) {
        return nullptr;
    }
    try {
        // whole 64-KiB (above 16 MiB whole 2-MiB) pieces, so that calls a
        // little larger than the last find their block again
        const std::size_t unit = bytes > (std::size_t{16} << 20) ? std::size_t{2} << 20
                                                                 : std::size_t{64} << 10;
        const std::size_t want = (std::max<std::size_t>(bytes, 1) + unit - 1) / unit * unit;
        {
            std::lock_guard<std::mutex> hold(g_mu);
            Block* best = nullptr;
            for (Block& b : g_blocks) {
                if (b.device == device && !b.busy && b.bytes >= want &&
                    b.bytes / kFitMost <= want &&
                    (best == nullptr || b.bytes < best->bytes)) {
                    best = &b;
                }
            }
            if (best != nullptr) {
                best->busy = true;
                return best->ptr;
            }
            g_blocks.reserve(g_blocks.size() + 1);
        }
        void* ptr = nullptr;
        if (hipMalloc(&ptr, want) != hipSuccess) {
            (void)hipGetLastError();
            scratch_trim();
            if (hipMalloc(&ptr, want) != hipSuccess) {
                (void)hipGetLastError();
                return nullptr;
            }
        }
        try {
            std::lock_guard<std::mutex> hold(g_mu);
            g_blocks.push_back(Block{ptr, want, device, true});
        } catch (const std::bad_alloc&) {
            (void)hipFree(ptr);
            return nullptr;
        }
        return ptr;
    } catch (const std::bad_alloc&) {
        return nullptr;
    }
}

void scratch_give(void* block)
{
    std::vector<void*> drop;
    try {
        std::lock_guard<std::mutex> hold(g_mu);
        for (std::size_t k = 0; k < g_blocks.size(); ++k) {
            if (g_blocks[k].ptr == block) {
                g_blocks[k].busy = false;
                // the block used last is the one kept longest
                std::rotate(g_blocks.begin() + static_cast<std::ptrdiff_t>(k),
                            g_blocks.begin() + static_cast<std::ptrdiff_t>(k) + 1,
                            g_blocks.end());
                drop = take_idle(g_blocks.back().device, kScratchKeep);
                break;
            }
        }
    } catch (const std::bad_alloc&) {
        // the block stays idle in the pool
    }
    for (void* p : drop) {
        (void)hipFree(p);
    }
}

void scratch_trim()
{
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) {
        return;
    }
    std::vector<void*> drop;
    try {
        std::lock_guard<std::mutex> hold(g_mu);
        drop = take_idle(device, 0);
    } catch (const std::bad_alloc&) {
    }
    for (void* p : drop) {
        (void)hipFree(p);
    }
}

void scratch_hold()
{
    std::lock_guard<std::mutex> hold(g_mu);
    ++g_holders;
}

void scratch_drop()
{
    std::vector<void*> drop;
    try {
        std::lock_guard<std::mutex> hold(g_mu);
        if (--g_holders == 0) {
            drop = take_idle(-1, 0);
        }
    } catch (const std::bad_alloc&) {
    }
    for (void* p : drop) {
        (void)hipFree(p);
    }
}

}  // namespace hbfamd
