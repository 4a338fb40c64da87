// Scratch device memory of an index build: ranges of a few large blocks.
//
// hipMalloc and hipFree of more than a few MB take 0.2 to 0.7 ms each, and a
// kd-tree build's arrays grow level by level: on the 199,713-triangle terrain
// 68 such calls were 24 ms of the 36 ms of an admission, its kernels 8 ms.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <map>
#include <string>
#include <vector>

#include "xt_device.h"

// Every range is used on d->stream alone, so one that is given back may be
// handed out again at once: the stream orders the uses. The blocks are freed,
// after the stream has drained, with the object. `exact`: every range is a
// block of its own that is freed when it is given back, so that no more is
// held than asked for (a build that does not fit the budget in large blocks
// is made again this way).
class XtScratch {
  public:
    XtScratch(xt_dev *dev, size_t block_bytes, bool exact_) : exact(exact_), d(dev), block(block_bytes) {}
    XtScratch(const XtScratch &) = delete;
    XtScratch &operator=(const XtScratch &) = delete;
    ~XtScratch() { release(); }
    // Every range back; the blocks are kept.
    void reset() {
        if (exact) return release();
        for (Block &b : blocks) b.free = {{0, b.bytes}};
    }
    // Every range back and the blocks freed.
    void release() {
        if (blocks.empty()) return;
        (void)hipStreamSynchronize(d->stream);
        for (Block &b : blocks) drop(b);
        blocks.clear();
    }
    const bool exact;

    // `bytes` rounded up to 256 device bytes, 256-aligned.
    int take(void **p, size_t bytes) {
        bytes = round(bytes);
        if (!exact)
            for (Block &b : blocks)
                for (auto it = b.free.begin(); it != b.free.end(); ++it)
                    if (it->second >= bytes) {
                        const size_t at = it->first, left = it->second - bytes;
                        b.free.erase(it);
                        if (left) b.free[at + bytes] = left;
                        *p = b.p + at;
                        return XT_OK;
                    }
        Block b;
        b.bytes = exact ? bytes : std::max(bytes, round(block));
        block = std::max<size_t>(block / 2, 1u << 20);
        if (d->budget && d->used + b.bytes > d->budget) b.bytes = bytes;
        if (d->budget && d->used + b.bytes > d->budget) {
            d->err = "device build exceeds the HBM budget";
            return XT_E_BUDGET;
        }
        const hipError_t e = hipMalloc((void **)&b.p, b.bytes);
        if (e != hipSuccess) {
            d->err = std::string("hipMalloc: ") + hipGetErrorString(e);
            (void)hipGetLastError();
            return exact ? XT_E_DEVICE : XT_E_BUDGET;
        }
        d->used += b.bytes;
        if (b.bytes > bytes) b.free[bytes] = b.bytes - bytes;
        *p = b.p;
        blocks.push_back(std::move(b));
        return XT_OK;
    }

    void give(void *p, size_t bytes) {
        bytes = round(bytes);
        for (size_t k = 0; k < blocks.size(); ++k) {
            Block &b = blocks[k];
            if ((char *)p < b.p || (char *)p >= b.p + b.bytes) continue;
            if (exact) {
                (void)hipStreamSynchronize(d->stream);
                drop(b);
                blocks.erase(blocks.begin() + (long)k);
                return;
            }
            auto it = b.free.emplace((size_t)((char *)p - b.p), bytes).first;
            auto nx = std::next(it);
            if (nx != b.free.end() && it->first + it->second == nx->first) {
                it->second += nx->second;
                b.free.erase(nx);
            }
            if (it != b.free.begin()) {
                auto pv = std::prev(it);
                if (pv->first + pv->second == it->first) {
                    pv->second += it->second;
                    b.free.erase(it);
                }
            }
            return;
        }
    }

    static size_t round(size_t bytes) { return (std::max<size_t>(bytes, 1) + 255) & ~(size_t)255; }

  private:
    struct Block {
        char *p = nullptr;
        size_t bytes = 0;
        std::map<size_t, size_t> free;  // offset -> bytes
    };
    void drop(Block &b) {
        (void)hipFree(b.p);
        d->used -= std::min<uint64_t>(d->used, b.bytes);
    }
    xt_dev *d;
    size_t block;  // bytes of the next block
    std::vector<Block> blocks;
};

// The first block of a scene's index builds: the kd-tree build of the terrain
// holds 420 bytes a primitive at its largest level, a wide BVH build 364.
inline size_t xt_build_block(uint32_t n_prims) { return 512ull * n_prims + (1u << 21); }
