// graph_input.load_from_csr on a GPU box, from host CSR arrays to every format on the device and on the host, as one native
// call.  What bounds it is PCIe: the CSR arrays go up, the 2x1 blocks and the row splits come down (143 and 230 MB for an
// R-MAT graph of 2^20 rows, 57 GB/s each way from page-locked memory).  Around the two transfers:
//   * the arrays are pageable (they are the caller's): worker threads copy them chunk by chunk into a ring of page-locked
//     slots and enqueue each slot's transfer (the runtime's own pageable path reaches 26 - 38 GB/s), and take the row
//     statistics between and after the copies;
//   * the values follow the indices on a stream of their own, while the blocks are counted, the row splits built and the
//     blocks' columns on their way back (the bus carries both directions at once);
//   * what needs the CPU stays off PyTorch's thread pool: its threads spin for milliseconds after a parallel operation and
//     held the workers up;
//   * three host waits instead of fourteen: counts, segments of the blocks' split, and the end.
// Step by step from Python the same work took 14 - 16 ms on that graph.
#pragma once
#include "glue_common.h"
#include <ATen/hip/HIPContext.h>
#include <atomic>
#include <cmath>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <mutex>
#include <thread>

namespace pspglue {

using torch::Tensor;

// ---- statistics of the rows (graph_input.py:60-87 of the reference), from exact integer sums -----------------------------
struct RowStats {
    long long occupied = 0, sum = 0, blocks_occupied = 0, sum_bw = 0;
    double sum2 = 0;  // of squared row lengths: exact below 2^53
    int max_nnz = 0, max_bw = 0;
    bool bad = false, any_width = false;
    void add(const RowStats &o)
    {
        occupied += o.occupied, sum += o.sum, blocks_occupied += o.blocks_occupied, sum_bw += o.sum_bw, sum2 += o.sum2;
        max_nnz = std::max(max_nnz, o.max_nnz);
        if (o.any_width) max_bw = any_width ? std::max(max_bw, o.max_bw) : o.max_bw;
        any_width = any_width || o.any_width;
        bad = bad || o.bad;
    }
};
// row lengths of the rows [r0, r1), r0 even
inline RowStats row_lengths(const int *rp, int *row_nnz, long long r0, long long r1, long long n, long long nnz)
{
    RowStats s;
    for (long long r = r0; r < r1; r++) {
        const int lo = rp[r], hi = rp[r + 1], k = hi - lo;
        if (lo > hi || lo < 0 || hi > nnz) s.bad = true;
        row_nnz[r] = k;
        if (k != 0) {
            s.occupied++, s.sum += k, s.sum2 += (double)k * (double)k;
            s.max_nnz = std::max(s.max_nnz, k);
        }
        if ((r & 1) == 0) s.blocks_occupied += rp[std::min(r + 2, n)] != lo;
    }
    return s;
}
// widths (last - first column) of the rows [r0, r1)
inline RowStats row_widths(const int *rp, const int *ci, long long r0, long long r1, long long nnz)
{
    RowStats s;
    for (long long r = r0; r < r1; r++) {
        const int lo = rp[r], hi = rp[r + 1];
        if (lo >= hi || lo < 0 || hi > nnz) continue;
        const int w = ci[hi - 1] - ci[lo];
        s.max_bw = s.any_width ? std::max(s.max_bw, w) : w;
        s.any_width = true;
        s.sum_bw += w;
    }
    return s;
}

// ---- host arrays to the device ---------------------------------------------------------------------------------------------
inline void hip_ok(hipError_t e) { TORCH_CHECK(e == hipSuccess, "HIP: ", hipGetErrorString(e)); }

// Work is a list in order: pieces of copies (kPiece bytes of a chunk each) and pieces of host work.  The worker threads take
// it from the front; the calling thread enqueues a chunk's transfer once its pieces are in the ring and frees the slot of the
// chunk before the last (few large transfers from one thread: with 2 MB transfers enqueued by the workers themselves the same
// arrays took twice as long).
class Uploader {
    static constexpr size_t kChunk = (size_t)8 << 20, kPiece = (size_t)1 << 20;
    static constexpr int kSlots = 16;  // the values wait in the ring for the indices to be up
    static constexpr int kWorkers = 6;  // copy some 100 GB/s between them, more than the bus takes
    struct Task {
        std::function<void()> work;  // host work, or:
        const char *src = nullptr;
        size_t bytes = 0, offset = 0;
        int chunk = -1, group = 0;
    };
    struct Chunk {
        char *dst;
        size_t bytes;
        hipStream_t stream;
    };
    std::vector<Task> tasks;
    std::vector<Chunk> chunks;
    std::vector<int> group_open, group_chunks;  // unfinished host tasks; one past the group's last chunk
    std::unique_ptr<std::atomic<int>[]> pieces;  // of every chunk, not yet in the ring
    std::atomic<size_t> next{0};
    std::atomic<int> slots_free{0};  // chunks below this may be written to the ring
    std::atomic<bool> stop{false};
    hipEvent_t events[kSlots] = {};
    Tensor ring;
    int device, enqueued = 0;
    std::mutex mu;
    std::condition_variable done;
    std::vector<std::thread> pool;

    void run_one(Task &t)
    {
        if (t.work) {
            t.work();
            std::lock_guard<std::mutex> lock(mu);
            if (--group_open[t.group] == 0) done.notify_all();
            return;
        }
        while (t.chunk >= slots_free.load(std::memory_order_acquire)) {
            if (stop) return;
            std::this_thread::yield();
        }
        std::memcpy((char *)ring.data_ptr() + (size_t)(t.chunk % kSlots) * kChunk + t.offset, t.src, t.bytes);
        pieces[t.chunk].fetch_sub(1, std::memory_order_release);
    }
    bool take_one()
    {
        const size_t i = next.fetch_add(1);
        if (i >= tasks.size()) return false;
        run_one(tasks[i]);
        return true;
    }
    // the calling thread helps, but takes nothing that waits for a slot only it can free
    bool help()
    {
        size_t i = next.load();
        if (i >= tasks.size() || tasks[i].chunk >= slots_free || !next.compare_exchange_strong(i, i + 1)) return false;
        run_one(tasks[i]);
        return true;
    }
    void enqueue_next()
    {
        const int c = enqueued;
        while (pieces[c].load(std::memory_order_acquire) != 0)
            if (!help()) std::this_thread::yield();
        const Chunk &k = chunks[c];
        hip_ok(hipMemcpyAsync(k.dst, (char *)ring.data_ptr() + (size_t)(c % kSlots) * kChunk, k.bytes, hipMemcpyHostToDevice, k.stream));
        enqueued++;
        // an event between two transfers costs some 40 us of the bus: only where a later chunk reuses the slot
        if (reused(c)) hip_ok(hipEventRecord(events[c % kSlots], k.stream));
        if (c >= 1 && reused(c - 1)) {  // two transfers stay queued
            hip_ok(hipEventSynchronize(events[(c - 1) % kSlots]));
            slots_free.store(c + kSlots, std::memory_order_release);
        }
    }

public:
    explicit Uploader(int device_) : device(device_) {}
    ~Uploader()
    {
        stop = true;
        for (auto &t : pool) t.join();
        // the ring is not given back while a transfer reads it
        hipStream_t last = nullptr;
        for (int c = 0; c < enqueued; c++)
            if (c == 0 || chunks[c].stream != last) (void)hipStreamSynchronize(last = chunks[c].stream);
        for (hipEvent_t e : events)
            if (e) (void)hipEventDestroy(e);
    }
    bool reused(int c) const { return c + kSlots < (int)chunks.size(); }
    int group()
    {
        group_open.push_back(0);
        group_chunks.push_back(0);
        return (int)group_open.size() - 1;
    }
    void copy(int g, const Tensor &src, Tensor &dst, hipStream_t stream)
    {
        const size_t total = src.nbytes();
        for (size_t o = 0; o < total; o += kChunk) {
            const size_t bytes = std::min(kChunk, total - o);
            for (size_t p = 0; p < bytes; p += kPiece) {
                Task t;
                t.src = (const char *)src.data_ptr() + o + p, t.bytes = std::min(kPiece, bytes - p), t.offset = p;
                t.chunk = (int)chunks.size(), t.group = g;
                tasks.push_back(std::move(t));
            }
            chunks.push_back({(char *)dst.data_ptr() + o, bytes, stream});
        }
        group_chunks[g] = (int)chunks.size();
    }
    void host_work(int g, std::function<void()> f)
    {
        Task t;
        t.work = std::move(f), t.group = g;
        tasks.push_back(std::move(t));
        group_open[g]++;
    }
    void start()
    {
        const int slots = std::min((int)chunks.size(), kSlots);
        if (slots > 0) ring = torch::empty({(long)(slots * kChunk)}, torch::TensorOptions().dtype(torch::kUInt8).pinned_memory(true));
        for (int i = 0; i < slots; i++) hip_ok(hipEventCreateWithFlags(&events[i], hipEventDisableTiming));
        pieces.reset(new std::atomic<int>[chunks.size() + 1]);
        for (size_t c = 0; c < chunks.size(); c++) pieces[c] = (int)((chunks[c].bytes + kPiece - 1) / kPiece);
        slots_free = kSlots;
        // a handful of pieces is done before threads have started
        const int workers = tasks.size() <= 8 ? 0 : kWorkers;
        for (int w = 0; w < workers; w++)
            pool.emplace_back([this] {
                while (!stop && take_one()) {}
            });
    }
    // the group's transfers are enqueued and its host work is done
    void wait(int g)
    {
        while (enqueued < group_chunks[g]) enqueue_next();
        std::unique_lock<std::mutex> lock(mu);
        while (group_open[g] != 0) {
            lock.unlock();
            const bool did = help();
            lock.lock();
            if (!did) break;
        }
        done.wait(lock, [&] { return group_open[g] == 0; });
    }
};

// one event per hand-over between the two streams
struct Event {
    hipEvent_t e = nullptr;
    Event() { hip_ok(hipEventCreateWithFlags(&e, hipEventDisableTiming)); }
    ~Event() { (void)hipEventDestroy(e); }
    void hand_over(hipStream_t from, hipStream_t to)
    {
        hip_ok(hipEventRecord(e, from));
        hip_ok(hipStreamWaitEvent(to, e, 0));
    }
};

// CSR arrays on the host -> formats.  The segment lengths of the row splits are the caller's rule: granularity(non-empty rows)
// for CSR, granularity_b(non-empty block-rows, blocks) for the 2x1 blocks.  flags: PSP_BUILD_* bits; with any set, only "flags" and the arrays of the CSR upload are valid.
inline py::dict load_formats(Tensor rowPtr, Tensor colIdx, Tensor val, long ncols, py::function granularity, py::function granularity_b)
{
    need_cpu(rowPtr, "rowPtr");
    need_cpu(colIdx, "colIdx");
    need_cpu(val, "val");
    need_i32(rowPtr, "rowPtr");
    need_i32(colIdx, "colIdx");
    need_f32(val, "val", 1);
    TORCH_CHECK(rowPtr.size(0) >= 2 && colIdx.size(0) == val.size(0), "load_formats: array sizes disagree");
    const long n = rowPtr.size(0) - 1, nnz = colIdx.size(0), nbr = (n + 1) / 2;
    const int device = (int)c10::hip::current_device();
    const auto dev_i = torch::TensorOptions().dtype(torch::kInt32).device(torch::kCUDA, device);
    const auto dev_f = dev_i.dtype(torch::kFloat32);
    const auto pin_i = torch::TensorOptions().dtype(torch::kInt32).pinned_memory(true);
    const auto pin_f = pin_i.dtype(torch::kFloat32);
    py::dict out;

    Tensor rp = torch::empty({n + 1}, dev_i), ci = torch::empty({nnz}, dev_i), v = torch::empty({nnz}, dev_f);
    Tensor row_nnz = torch::empty({n}, torch::kInt32);
    const hipStream_t main = (hipStream_t)stream_of(rp);
    auto side_stream = c10::hip::getStreamFromPool(false, device);
    const hipStream_t side = side_stream.stream();
    Event ev0, ev1;
    ev0.hand_over(main, side);  // the memory of `v` may have had a use on this stream

    RowStats st;
    std::mutex st_mu;
    Uploader up(device);
    const int g_rows = up.group(), g_index = up.group(), g_rest = up.group();
    const int *rph = rowPtr.data_ptr<int>(), *cih = colIdx.data_ptr<int>();
    int *kh = row_nnz.data_ptr<int>();
    const long piece = 1 << 16;
    up.copy(g_index, rowPtr, rp, main);
    up.copy(g_index, colIdx, ci, main);
    for (long r = 0; r < n; r += piece)
        up.host_work(g_rows, [&, r] {
            RowStats s = row_lengths(rph, kh, r, std::min(r + piece, n), n, nnz);
            std::lock_guard<std::mutex> lock(st_mu);
            st.add(s);
        });
    up.copy(g_rest, val, v, side);
    for (long r = 0; r < n; r += piece)
        up.host_work(g_rest, [&, r] {
            RowStats s = row_widths(rph, cih, r, std::min(r + piece, n), nnz);
            std::lock_guard<std::mutex> lock(st_mu);
            st.add(s);
        });
    up.start();

    // counts: blocks per block-row, segments per row
    Tensor rpb = torch::empty({nbr + 1}, dev_i), seg = torch::empty({n + 1}, dev_i), status = torch::zeros({2}, dev_i);
    const int ws_ints = psp_scan_workspace_ints((int)n);
    Tensor ws = torch::empty({ws_ints}, dev_i), counts = torch::empty({8}, pin_i);
    int *counts_h = counts.data_ptr<int>(), *status_d = status.data_ptr<int>();
    up.wait(g_index);
    up.wait(g_rows);
    double occupied;
    {
        std::lock_guard<std::mutex> lock(st_mu);
        if (st.bad || rph[0] != 0 || rph[n] != nnz) {
            out["flags"] = (int)PSP_BUILD_BAD_ROWPTR;
            return out;
        }
        occupied = (double)st.occupied;
    }
    const int g = granularity(st.occupied).cast<int>();
    TORCH_CHECK(g >= 1, "split_granularity must be positive");
    ok(psp_check_index_dev(ip(rp), ip(ci), nullptr, (int)n, (int)nnz, (int)ncols, 0, status_d, main));
    ok(psp_bcsr_offsets_dev(ip(rp), ip(ci), (int)n, rpb.data_ptr<int>(), ws.data_ptr<int>(), ws_ints, status_d, main));
    ok(psp_split_csr_offsets_dev(ip(rp), (int)n, g, seg.data_ptr<int>(), ws.data_ptr<int>(), ws_ints, status_d, main));
    auto fetch = [&](int slot, const int *from) { hip_ok(hipMemcpyAsync(counts_h + slot, from, 4, hipMemcpyDeviceToHost, main)); };
    fetch(0, status_d);
    fetch(1, ip(rpb) + nbr);
    fetch(2, ip(seg) + n);
    hip_ok(hipStreamSynchronize(main));
    const int flags = counts_h[0];
    const long nblk = counts_h[1], S = counts_h[2];
    out["rowPtr"] = rp;
    out["colIdx"] = ci;
    out["val"] = v;
    if (flags) {
        up.wait(g_rest);
        ev1.hand_over(side, main);
        hip_ok(hipStreamSynchronize(main));
        out["flags"] = flags;
        return out;
    }

    // row split of the CSR arrays, segments of the blocks' split
    const int gb = granularity_b(st.blocks_occupied, nblk).cast<int>();
    TORCH_CHECK(gb >= 1, "split_granularity must be positive");
    Tensor rps = torch::empty({S + 1}, dev_i), tr = torch::empty({S}, dev_i), segb = torch::empty({nbr + 1}, dev_i);
    ok(psp_split_csr_fill_dev(ip(rp), ip(seg), (int)n, g, (int)S, rps.data_ptr<int>(), tr.data_ptr<int>(), main));
    ok(psp_split_csr_offsets_dev(ip(rpb), (int)nbr, gb, segb.data_ptr<int>(), ws.data_ptr<int>(), ws_ints, status_d + 1, main));
    fetch(3, ip(segb) + nbr);
    fetch(4, status_d + 1);
    hip_ok(hipStreamSynchronize(main));
    TORCH_CHECK(counts_h[4] == 0, "load_formats: the blocks' row pointer is inconsistent");
    const long Sb = counts_h[3];
    Tensor cib = torch::empty({nblk}, dev_i), vb = torch::empty({nblk, 2}, dev_f);
    ok(psp_bcsr_fill_dev(ip(rp), ip(ci), nullptr, (int)n, ip(rpb), cib.data_ptr<int>(), nullptr, main));
    Tensor rpbs = torch::empty({Sb + 1}, dev_i), trb = torch::empty({Sb}, dev_i);
    ok(psp_split_csr_fill_dev(ip(rpb), ip(segb), (int)nbr, gb, (int)Sb, rpbs.data_ptr<int>(), trb.data_ptr<int>(), main));

    auto to_host = [&](const Tensor &d, const torch::TensorOptions &o) {
        Tensor h = torch::empty(d.sizes(), o);
        if (d.numel()) hip_ok(hipMemcpyAsync(h.data_ptr(), d.data_ptr(), d.nbytes(), hipMemcpyDeviceToHost, main));
        return h;
    };
    Tensor h_rps = to_host(rps, pin_i), h_tr = to_host(tr, pin_i), h_rpb = to_host(rpb, pin_i), h_rpbs = to_host(rpbs, pin_i),
           h_trb = to_host(trb, pin_i), h_cib = to_host(cib, pin_i);
    up.wait(g_rest);
    ev1.hand_over(side, main);
    hip_ok(hipEventRecord(ev0.e, main));  // the index arrays are down: h_rpb is read below
    ok(psp_bcsr_fill_dev(ip(rp), ip(ci), fp(v), (int)n, ip(rpb), nullptr, fpw(vb), main));
    Tensor h_vb = to_host(vb, pin_f);

    // meanwhile: the statistics as the caller wants them
    Tensor row_nnz_b = torch::empty({nbr}, torch::kInt32), split_nnz = torch::empty({n}, torch::kFloat32),
           split_nnz_b = torch::empty({nbr}, torch::kFloat32);
    hip_ok(hipEventSynchronize(ev0.e));
    const int *rpbh = h_rpb.data_ptr<int>();
    int *kbh = row_nnz_b.data_ptr<int>();
    for (long t = 0; t < nbr; t++) kbh[t] = rpbh[t + 1] - rpbh[t];
    auto segments = [](const int *k, float *f, long m, int len) {
        for (long i = 0; i < m; i++) f[i] = std::ceil((float)k[i] / (float)len);
    };
    segments(kh, split_nnz.data_ptr<float>(), n, g);
    segments(kbh, split_nnz_b.data_ptr<float>(), nbr, gb);
    const double var_all = n > 1 ? (st.sum2 - (double)st.sum * (double)st.sum / (double)n) / (double)(n - 1) : NAN;
    const double var_occ = occupied > 1 ? (st.sum2 - (double)st.sum * (double)st.sum / occupied) / (occupied - 1) : NAN;
    out["flags"] = 0;
    out["row_nnz"] = row_nnz;
    out["max_row_nnz"] = st.max_nnz;
    out["real_nrow"] = st.occupied;
    out["std"] = std::sqrt(std::max(var_all, 0.0));
    out["std_occupied"] = std::sqrt(std::max(var_occ, 0.0));
    out["max_bw"] = st.max_bw;
    out["sum_bw"] = st.sum_bw;
    out["blocks_stats"] = py::make_tuple(row_nnz_b, st.blocks_occupied, gb, Sb, split_nnz_b);
    out["split_stats"] = py::make_tuple(g, S, split_nnz);
    hip_ok(hipStreamSynchronize(main));
    out["split"] = std::vector<Tensor>{rps, tr, h_rps, h_tr};
    out["blocks"] = std::vector<Tensor>{rpb, cib, vb, h_rpb, h_cib, h_vb};
    out["blocks_split"] = std::vector<Tensor>{rpbs, trb, h_rpbs, h_trb};
    return out;
}

}  // namespace pspglue
