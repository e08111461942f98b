// Copies between the caller's ordinary host memory and the device.
//
// The runtime moves ordinary (pageable) memory at 26 GB/s up and 16 GB/s down on this machine; from
// and to pinned memory the link gives 54 GB/s, and one thread copies between the two kinds at
// 30 GB/s.  So a transfer goes through a pinned buffer in pieces, the host's part of a piece under
// the link's part of another.  Pieces of 2 MiB: every piece costs some 8 us of the runtime's time
// (256 KiB: 527 us for 9.8 MB up, 512 KiB 358, 1 MiB 288, 2 MiB 260, 4 MiB 277, one piece 336; the
// runtime's own path 390).  Down, a few threads share the host's part (7.4 MB: 430 us with one
// thread, 265 with two, 244 with four; the runtime's own path 450); up they do not pay, because
// nothing can start before they have (260 against 280 to 330).
#include <atomic>
#include <cstring>
#include <exception>
#include <thread>

#include "preprocess.h"

namespace accel {

// All queue on s and return when the host's side is done: upload when src has been read (the copy
// to dst is ordered on s), download and download_made when dst has been written.
int upload(void *dst, const void *src, size_t bytes, hipStream_t s)
{
    StageHolder st(bytes);
    if (!st.s) return ACCEL_ERR_ALLOC;
    for (size_t off = 0; off < bytes; off += kStagePiece) {
        const size_t at = off % kStageBytes, n = std::min(bytes - off, kStagePiece);
        const hipEvent_t done = st.s->event[at / kStagePiece];      // behind the last copy out of this piece
        if (off >= kStageBytes) ACCEL_HIP(hipEventSynchronize(done));
        char *stage = static_cast<char *>(st.s->p) + at;
        memcpy(stage, static_cast<const char *>(src) + off, n);
        st.s->in_doubt = true;
        ACCEL_HIP(hipMemcpyAsync(static_cast<char *>(dst) + off, stage, n, hipMemcpyHostToDevice, s));
        if (bytes > kStageBytes) ACCEL_HIP(hipEventRecord(done, s));
    }
    ACCEL_HIP(hipEventRecord(st.s->last, s));           // who takes the buffer next waits for its last copy
    st.s->busy = true;
    st.s->in_doubt = false;
    return ACCEL_OK;
}

static int copy_piece(const void *src, void *stage, size_t offset, size_t bytes, hipStream_t s)
{
    ACCEL_HIP(hipMemcpyAsync(stage, static_cast<const char *>(src) + offset, bytes, hipMemcpyDeviceToHost, s));
    return ACCEL_OK;
}

int download(void *dst, const void *src, size_t bytes, hipStream_t s)
{
    return download_made(dst, bytes, s, copy_piece, src);
}

int download_made(void *dst, size_t bytes, hipStream_t s, MakePiece make, const void *context)
{
    StageHolder st(bytes);
    if (!st.s) return ACCEL_ERR_ALLOC;
    for (size_t done = 0; done < bytes;) {
        const size_t here = std::min(bytes - done, kStageBytes);
        const int n = (int)((here + kStagePiece - 1) / kStagePiece);
        st.s->in_doubt = true;
        char *to = static_cast<char *>(dst) + done, *stage = static_cast<char *>(st.s->p);
        for (int i = 0; i < n; i++) {
            const size_t off = (size_t)i * kStagePiece;
            if (int rc = make(context, stage + off, done + off, std::min(kStagePiece, here - off), s)) return rc;
            ACCEL_HIP(hipEventRecord(st.s->event[i], s));
        }
        std::atomic<int> next{0}, arrived{0};
        auto copy_pieces = [&]() {
            for (int i; (i = next.fetch_add(1)) < n;) {
                while (arrived.load(std::memory_order_acquire) <= i) std::this_thread::yield();
                const size_t off = (size_t)i * kStagePiece;
                memcpy(to + off, stage + off, std::min(kStagePiece, here - off));
            }
        };
        // helpers start while the first pieces are on the link; none for a single piece
        constexpr int kHelpers = 3;
        std::thread helper[kHelpers];
        int n_helpers = 0;
        try {
            for (; n_helpers < std::min(kHelpers, n - 1); n_helpers++) helper[n_helpers] = std::thread(copy_pieces);
        } catch (const std::exception &) {              // no thread or no memory for one: fewer, then
        }
        hipError_t e = hipSuccess;
        for (int i = 0; i < n; i++) {
            if (e == hipSuccess) e = hipEventSynchronize(st.s->event[i]);
            arrived.store(i + 1, std::memory_order_release);        // (after an error too: the helpers have to end)
        }
        copy_pieces();
        for (int i = 0; i < n_helpers; i++) helper[i].join();
        ACCEL_HIP(e);
        st.s->in_doubt = false;
        done += here;
    }
    return ACCEL_OK;
}

}  // namespace accel
