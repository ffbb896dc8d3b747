// Pinned host memory that the threads of one context share.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <deque>
#include <memory>
#include <mutex>
#include <vector>

namespace nxm {

// Chunks of pinned host memory.  A scene staged for upload on one thread
// (nxm_scene_stage_upload) holds a chunk until the thread that steps its world has queued the
// copies and seen them done (PendingUploads); a readback holds one for its own call.  A
// chunk that is not held has nothing queued on it: taking one asks no event and no stream,
// whichever of them are being captured or gone.
class PinnedPool {
  public:
    PinnedPool() = default;
    PinnedPool(const PinnedPool &) = delete;
    PinnedPool &operator=(const PinnedPool &) = delete;
    ~PinnedPool()
    {
        for (auto &c : chunks_) (void)hipHostFree(c.p);
    }

    // The smallest free chunk of at least `bytes`.
    hipError_t take(size_t bytes, int *idx, char **out)
    {
        std::lock_guard<std::mutex> g(mu_);
        int best = -1;
        for (int k = 0; k < (int)chunks_.size(); ++k)
            if (!chunks_[k].held && chunks_[k].n >= bytes && (best < 0 || chunks_[k].n < chunks_[best].n)) best = k;
        if (best < 0) {
            Chunk c;
            c.n = std::max<size_t>(bytes, (size_t)1 << 20);
            const hipError_t e = hipHostMalloc(reinterpret_cast<void **>(&c.p), c.n, hipHostMallocDefault);
            if (e != hipSuccess) return e;
            chunks_.push_back(c);
            best = (int)chunks_.size() - 1;
        }
        chunks_[best].held = true;
        *idx = best;
        *out = chunks_[best].p;
        return hipSuccess;
    }
    // Gives a chunk back on which nothing is queued any more.
    void give(int idx)
    {
        std::lock_guard<std::mutex> g(mu_);
        chunks_[idx].held = false;
    }
    char *ptr(int idx)
    {
        std::lock_guard<std::mutex> g(mu_);
        return chunks_[idx].p;
    }

  private:
    struct Chunk {
        char *p = nullptr;
        size_t n = 0;
        bool held = false;
    };
    std::mutex mu_;
    std::vector<Chunk> chunks_;
};

// The chunks whose copies one world has queued on its stream, in order, used by the thread
// that steps the world: the events are its own, recorded and asked for outside captures and
// never after the stream.
class PendingUploads {
  public:
    ~PendingUploads()
    {
        drain();
        for (hipEvent_t e : spare_) (void)hipEventDestroy(e);
    }

    // Takes over a held chunk of the pool whose copies have just been queued on st.
    hipError_t add(std::shared_ptr<PinnedPool> pool, int chunk, hipStream_t st)
    {
        hipEvent_t ev = nullptr;
        hipError_t e = hipSuccess;
        if (!spare_.empty()) {
            ev = spare_.back();
            spare_.pop_back();
        } else {
            e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        }
        if (e == hipSuccess) {
            e = hipEventRecord(ev, st);
            if (e != hipSuccess) spare_.push_back(ev);
        }
        if (e != hipSuccess) {
            (void)hipStreamSynchronize(st);   // no event to wait for
            pool->give(chunk);
            return e;
        }
        list_.push_back(Upload{std::move(pool), chunk, ev});
        return hipSuccess;
    }
    // Gives back the chunks whose copies are done.
    hipError_t poll()
    {
        while (!list_.empty()) {
            const hipError_t e = hipEventQuery(list_.front().ev);
            if (e == hipErrorNotReady) break;
            if (e != hipSuccess) return e;
            release();
        }
        return hipSuccess;
    }
    // Gives back every chunk: the stream has been synchronized since their copies.
    void drain()
    {
        while (!list_.empty()) release();
    }

  private:
    struct Upload {
        std::shared_ptr<PinnedPool> pool;   // (the scene's context may go before the world)
        int chunk;
        hipEvent_t ev;
    };
    void release()
    {
        Upload &u = list_.front();
        u.pool->give(u.chunk);
        spare_.push_back(u.ev);
        list_.pop_front();
    }
    std::deque<Upload> list_;
    std::vector<hipEvent_t> spare_;
};

}  // namespace nxm
