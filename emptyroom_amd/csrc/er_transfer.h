// er_transfer.h -- copies between the caller's pageable memory and the device.
//
// The runtime stages a pageable copy on one thread, which also takes every page
// fault of a fresh array, and some small ones very slowly: a 41 MB grid into a
// fresh array took 4.05 ms where the link (56 GB/s) needs 0.73, 0.5 MB 0.22 ms.
// A Transfer copies through pinned memory of its own: up to 1 MiB through one
// small buffer, larger results through a ring of slots that the link fills while
// the caller, and for large arrays three threads, copy others to the array.
// Download, runtime / Transfer: 256 KiB 117 / 21 us, 512 KiB 225 / 41, 4 MiB 250 /
// 156, 16 MiB 970 / 630, 64 MiB 6640 / 2240, 256 MiB 25700 / 7260.  Uploads above
// 1 MiB reach 30 GB/s by the runtime's own path, which they keep.
//
// The contexts of a device share one Transfer (the pinned memory, 19 MiB at
// most, and the threads are made by the first copy that uses them and given back
// with the last context).  One copy at a time uses it; a copy that finds it in
// use takes the runtime's path.  The ring is taken when the stream has ended what is
// before the copy, so neither it nor a core is held while a kernel runs.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

#include <atomic>
#include <condition_variable>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace er {

class Transfer {
  public:
    static std::shared_ptr<Transfer> of_device(int device);
    ~Transfer();
    // dev -> host on stream s, after what s holds; returns when the bytes are in
    // host memory.
    hipError_t out(void *host, const void *dev, size_t bytes, hipStream_t s);
    // Holds the small buffer of an upload until its stream has passed it (no event does:
    // one that outlives the stream it was recorded on cannot be waited for).  The holder
    // makes no other call of this class.
    class Staged {
      public:
        ~Staged();

      private:
        friend class Transfer;
        std::unique_lock<std::mutex> lk_;
        hipStream_t s_ = nullptr;
    };
    // host -> dev on stream s, through the small buffer if that is free; host
    // memory must stay until s has passed the copy, and so must *hold.
    hipError_t in(void *dev, const void *host, size_t bytes, hipStream_t s, Staged *hold);
    // The small buffer (kBuffer bytes, device-accessible) for as long as the lock
    // is held; *p = nullptr if it is in use or cannot be had.
    std::unique_lock<std::mutex> small(char **p);
    static constexpr size_t kSmall = 1 << 20;   // bytes it is used for by copies, at most
    static constexpr size_t kBuffer = 3 << 20;

  private:
    struct Job;
    bool ensure(long chunks, bool threads);
    void start(Job *job);
    void finish();
    void work();
    std::mutex busy_;               // held by the copy that uses what follows
    char *small_ = nullptr;
    std::vector<char *> slot_;      // pinned, one size
    std::vector<std::thread> threads_;
    std::mutex mu_;                 // guards what follows
    std::condition_variable cv_;
    Job *job_ = nullptr;            // the copy to help with
    unsigned long count_ = 0;       // copies helped with
    int active_ = 0;                // threads helping
    bool stop_ = false;
};

}  // namespace er
