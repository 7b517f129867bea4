// HIP kernels of the tiled Cholesky library (gfx950).
#include <algorithm>

#include "kernels.hpp"
#include "executor.hpp"

namespace ttad {

// ---------------------------------------------------------------------------
// Host-sequenced executor: one block per work item of a batch of tasks.
// prefix[t] = first global item of task t (exclusive scan of n_items).
// ---------------------------------------------------------------------------
template <int VM>
__global__ __launch_bounds__(NTHREADS, vset_occupancy(VM)) void k_items(const DevMat* mats, const DevTask* tasks, const int32_t* prefix,
                                                    int n_tasks, int32_t* err) {
    extern __shared__ __align__(16) char lds[];
    const int g = blockIdx.x;
    int lo = 0, hi = n_tasks - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (prefix[mid] <= g) lo = mid;
        else hi = mid - 1;
    }
    const DevTask t = tasks[lo];
    // POTRF items wait only on lower-numbered blocks of the same launch, which are
    // dispatched first
    if (!exec_item<VM>(t, g - prefix[lo], mats, lds, err, (int64_t)500000000) && threadIdx.x == 0) atomicCAS(err, 0, 3);
}

// ---------------------------------------------------------------------------
// Persistent DAG executor (replaces the Threadpool worker loop). Work queues are ordered
// by priority; a queue is either shared or homed on one XCD (the GEMM/SYRK items of a
// priority bucket are split by output tile row, so that the items of one tile update,
// and the updates that share its A operand, meet in one XCD's L2). Every workgroup loops:
//   wave 0 reads the heads/tails of the queues 64 at a time (one per lane) and claims
//   the head entry of the first non-empty queue that is shared or homed on its own XCD;
//   when there is none it takes the first non-empty queue of another XCD (stealing).
//   A claim takes one credit from the queue's count of unclaimed entries (fetch-add -1;
//   a claimer that finds none gives it back) and then its slot (fetch-add on the head):
//   the credits never exceed the pushed entries, so a slot never passes the tail, and
//   no claim retries a compare-and-swap (CAS claims near the tail, with hundreds of
//   workers on few queues, cost more than half the executor's time in measurements).
//   The workgroup runs that work item, then thread 0 decrements the
//   task's remaining-items counter; the last item of a task decrements its
//   successors' dependency counters and pushes every item of a successor that
//   reaches zero into its queue. A worker exits when every item is done, or claimed by others.
// Memory ordering: item outputs are released (agent scope) before the counter
// RMWs; queue entries are written and polled relaxed, behind that release and in front of
// an acquire fence, so a consumer on another XCD sees the producer's tiles.
// The loop also ends when the abort flag is raised (watchdog: no work found for
// spin_limit ticks; queue overflow; an item variant missing from this instantiation).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void push_task(const DevGraph& g, const DevEdge& t) {
    const int b = t.bucket;
    const int pos = __hip_atomic_fetch_add(g.q_tail + b, t.n_items, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (pos + t.n_items > t.cap) {
        __hip_atomic_store(g.abort_flag, 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    // the caller's release fence orders these entries after the outputs they announce
    for (int r = 0; r < t.n_items; r++)
        __hip_atomic_store(g.q_items + t.base + pos + r, ((int64_t)t.succ << 20) | r, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    // claim credits (a claimer that gets a slot whose entry is not written yet polls it)
    __hip_atomic_fetch_add(g.q_count + b, t.n_items, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int VM>
__global__ __launch_bounds__(NTHREADS, vset_occupancy(VM)) void k_persistent(DevGraph g) {
    extern __shared__ __align__(16) char lds[];
    __shared__ int64_t s_item;
    const int tid = threadIdx.x;
    const int my_xcd = xcc_id();
    // The first worker started on a CU is its primary. A secondary (the second workgroup on that
    // CU) only takes items from a queue that holds more than there are idle primaries, so that
    // scarce work spreads one item per CU instead of pairing up on some CUs while others idle.
    __shared__ int s_primary, s_key;
    if (tid == 0) {
        s_key = cu_key();
        s_primary = __hip_atomic_fetch_add(g.cu_slots + s_key, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0;
    }
    __syncthreads();
    const bool primary = s_primary != 0;
    const int my_key = s_key;
    // idle primaries are counted per XCD (counters 256 bytes apart): the queues a worker mostly claims
    // from are those of its XCD
    int32_t* idle_primary = g.idle_primary + my_xcd * 64;
    if (primary && tid == 0) __hip_atomic_fetch_add(idle_primary, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    uint32_t rng = blockIdx.x * 2654435761u + 0x9e3779b9u;
    const int own_q = homed_queue(my_xcd, 0);  // first queue homed on this XCD
    for (;;) {
        if (tid < 64) {
            // wave 0, lane = priority bucket (highest first): the bucket's shared queue and the one homed on
            // this XCD. Each scan reads the two (their counters lie in 256-byte blocks that only the workers
            // of one XCD hammer) in one memory round trip; the other XCDs' queues only when both are empty.
            int64_t got = -1;
            int idle_scans = 0, done_before = -1;
            const int64_t t_start = (int64_t)wall_clock64();
            for (;;) {
                int cand[CLAIM_TRIES];  // queues to try, best first
                int nc = 0;
                int reserve_all = 0, reserve_own = 0;
                // From its third look on, a secondary does not even scan while a quarter of its XCD's primaries look for
                // work. (From the first idle primary on, bf16x3 factorization n = 32768: 66.8 ms, since an idle primary may be
                // held back by a critical item of its CU; from 8 on 57.1, from 16 on 57.2; n = 16384: 10.1, 10.9, 11.2 ms.
                // Primaries between two short tasks count as idle too: 2e5 independent empty tasks 16.2 ms held back from the
                // first look on, 11.4 so, 15.9 from the second; factorizations alike.)
                if (primary || idle_scans < 2 || ld_relaxed(idle_primary) < IDLE_PRIMARIES) {
                    // a secondary leaves queues that the idle primaries can drain; nothing is taken while
                    // the other worker of this CU runs an item of the critical path
                    // the lane index, opaque to the compiler here: addresses derived from it are formed per scan
                    // instead of being hoisted out of the worker loop, where they would hold registers through
                    // every item
                    int lane = tid;
                    asm volatile("" : "+v"(lane));
                    // (idle primaries of this XCD for its own queues, of all XCDs for shared queues and stealing)
                    int idle[NXCD];
#pragma unroll
                    for (int x = 0; x < NXCD; x++) idle[x] = primary ? 0 : ld_relaxed(g.idle_primary + x * 64);
                    const bool blocked = ld_relaxed(g.cu_crit + my_key) != 0;
                    const int cs = ld_relaxed(g.q_count + shared_queue(lane)), co = ld_relaxed(g.q_count + own_q + lane);
#pragma unroll
                    for (int x = 0; x < NXCD; x++) {
                        reserve_all += idle[x];
                        if (x == my_xcd) reserve_own = idle[x];
                    }
                    const unsigned long long ms = __ballot(!blocked && cs > reserve_all);
                    const unsigned long long mo = __ballot(!blocked && co > reserve_own);
                    // within a bucket the shared queue (POTRF, TRSM, FP64 updates) comes first
                    for (unsigned long long m = ms | mo; m != 0 && nc < CLAIM_TRIES; m &= m - 1) {
                        const int b = __ffsll((long long)m) - 1;
                        if ((ms >> b) & 1) cand[nc++] = shared_queue(b);
                        if (nc < CLAIM_TRIES && ((mo >> b) & 1)) cand[nc++] = own_q + b;
                    }
                    if (nc == 0 && !blocked) {  // nothing on this XCD: steal from the best bucket of another one
                        int cx[NXCD];
#pragma unroll
                        for (int x = 0; x < NXCD; x++) cx[x] = ld_relaxed(g.q_count + homed_queue(x, lane));
                        unsigned long long mx[NXCD], any = 0;
#pragma unroll
                        for (int x = 0; x < NXCD; x++) {
                            mx[x] = x == my_xcd ? 0ull : __ballot(cx[x] > reserve_all);
                            any |= mx[x];
                        }
                        if (any) {
                            const int b = __ffsll((long long)any) - 1;
#pragma unroll
                            for (int d = 1; d < NXCD; d++) {  // from the next XCD on, so that stealers spread
                                const int x = (my_xcd + d) % NXCD;
                                if (nc < CLAIM_TRIES && ((mx[x] >> b) & 1)) cand[nc++] = homed_queue(x, b);
                            }
                        }
                    }
                }
                if (nc > 0) {
                    int64_t e = -1;
                    if (tid == 0) {
                        int slot = -1, fb = -1;
                        // a credit lost to another worker: the next candidate at once (one atomic) rather than
                        // a new scan
                        for (int c = 0; c < nc; c++) {
                            const int b = cand[c];
                            const int reserve = b >= own_q && b < own_q + QUEUE_BUCKETS ? reserve_own : reserve_all;
                            if (__hip_atomic_fetch_add(g.q_count + b, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >
                                reserve) {
                                slot = __hip_atomic_fetch_add(g.q_head + b, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                                fb = b;
                                break;
                            }
                            // no credit left for this worker: give it back
                            __hip_atomic_fetch_add(g.q_count + b, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        }
                        if (slot >= 0) {
                            const int64_t* sp = g.q_items + g.q_base[fb] + slot;
                            // claimed before its producer wrote it: poll relaxed (an acquire load would
                            // invalidate the L2 on every poll); the acquire fence follows the broadcast
                            while ((e = ld_relaxed64(sp)) < 0) {
                                if ((int64_t)wall_clock64() - t_start > g.spin_limit) {
                                    __hip_atomic_store(g.abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                                    e = -2;
                                    break;
                                }
                                __builtin_amdgcn_s_sleep(1);
                            }
                        }
                    }
                    e = __shfl(e, 0);
                    if (e >= 0 || e == -2) {
                        got = e;
                        break;
                    }
                    // lost the race for the last credits: back off a random 0-15 x 64 cycles so the losers do
                    // not retry in lockstep
                    rng = rng * 1664525u + 1013904223u;
                    for (uint32_t q = rng >> 28; q > 0; q--) __builtin_amdgcn_s_sleep(1);
                    continue;
                }
                // every item done (or the run stopped): this worker is done
                const int done = ld_relaxed(g.done_items);
                if (done == g.total_items || ld_relaxed(g.abort_flag) != 0) {
                    got = -2;
                    break;
                }
                // So it is once every item is claimed: nothing will come, however long the last items still run, and its CU
                // is free for other work. The queues' heads are only looked at where that is likely, no task having
                // finished since the last look after a longest pause, and before the watchdog is raised.
                const bool expired = (int64_t)wall_clock64() - t_start > g.spin_limit;
                if (expired || (idle_scans == IDLE_BACKOFF && done == done_before)) {
                    int lane = tid;  // (opaque, as above)
                    asm volatile("" : "+v"(lane));
                    bool open = false;  // this lane's bucket: the shared queue, the homed ones
#pragma unroll 1
                    for (int x = 0; x <= NXCD; x++) {
                        const int q = x == NXCD ? shared_queue(lane) : homed_queue(x, lane);
                        open |= ld_relaxed(g.q_head + q) < g.q_base[q + 1] - g.q_base[q];
                    }
                    const bool any_open = __ballot(open) != 0;
                    if (expired && any_open && tid == 0)
                        __hip_atomic_store(g.abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (expired || !any_open) {
                        got = -2;
                        break;
                    }
                }
                done_before = done;
                // Idle workers look less often the longer they find nothing (a random 0 .. 2^k - 1 units of 64 cycles,
                // k up to IDLE_BACKOFF): with hundreds of them idle the next item still meets a scanner within
                // a fraction of a microsecond, and their loads no longer slow the claims and counters of the few
                // workers on the critical path. Pauses of up to 2^2 / 2^8 / 2^10 units, bf16x3 factorization n = 16384:
                // 12.1 / 10.4 / 10.2 ms; FP64 n = 2048 b = 256: 1.50 / 1.34 / 1.28 ms.
                idle_scans = min(idle_scans + 1, IDLE_BACKOFF);
                rng = rng * 1664525u + 1013904223u;
                for (uint32_t q = rng >> (32 - idle_scans); q > 0; q--) __builtin_amdgcn_s_sleep(1);
            }
            if (tid == 0) {
                s_item = got;
                if (primary && got >= 0)
                    __hip_atomic_fetch_add(idle_primary, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        __syncthreads();
        const int64_t e = s_item;
        if (e < 0) break;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        // the entry is the same for the whole workgroup (read from LDS): scalar registers, so that the task
        // record, its tiles and every size derived from them are scalar and their branches uniform
        const int task = __builtin_amdgcn_readfirstlane((int)(e >> 20));
        const int item = __builtin_amdgcn_readfirstlane((int)(e & 0xFFFFF));
        const DevTask t = g.tasks[task];
        const GemmOperands* go = g.gops + (long)task * g.gop_stride;  // (GEMM/SYRK items use them)
        if (tid == 0) {
            if (t.crit) __hip_atomic_fetch_add(g.cu_crit + my_key, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_fetch_add(g.xcd_run + (long)task * NXCD + my_xcd, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        uint64_t t0 = 0;
        if (g.trace && tid == 0) t0 = wall_clock64();
        const bool ran = exec_item<VM, true>(t, item, g.mats, lds, g.abort_flag, g.spin_limit, go);
        // Every wave waits until the L2 has acknowledged its own stores (gfx9: vmcnt counts stores too;
        // encoding vmcnt(0) expcnt(7) lgkmcnt(15)) before the barrier: after it, thread 0's decrement
        // below is issued only once all of this item's outputs sit in this XCD's L2.
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
        if (tid < 64) {
            int left = 0;
            uint64_t t1 = 0;
            // The task record is read again (its fields would hold registers through the item: the FP64 loop then spills)
            // and this lane's out-edge, both on their way while the counters below are updated.
            int task_again = task;
            asm volatile("" : "+s"(task_again));
            const DevTask tc = g.tasks[task_again];
            DevEdge ed{};
            if (tid < tc.edge_cnt) ed = g.edges[tc.edge_off + tid];
            if (tid == 0) {
                // Release elision: an agent-scope release (buffer_wbl2) writes back every dirty line of this
                // XCD's L2, so the item that leaves no other item of its task running on this XCD releases for
                // all of them; the others skip it. This relies on the hardware, not on the memory model: an
                // item's stores reached the L2 before its relaxed decrement was issued (the wait above), the
                // decrements of one counter are serialized at the L2, and the last one's write-back is issued
                // after its decrement returned, so it covers every earlier item's lines. Each item decrements
                // the task's remaining count after that, so the count reaches zero only after every XCD that
                // ran items of the task has released.
                if (__hip_atomic_fetch_add(g.xcd_run + (long)task * NXCD + my_xcd, -1, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT) == 1)
                    release_agent();
                if (!ran) __hip_atomic_store(g.abort_flag, 3, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (g.trace) t1 = wall_clock64();
                // Counters are relaxed: the release above has written this item's outputs back before the decrement.
                // The wave that takes a counter to zero acquires what the other decrements released; it has nothing
                // of its own left to write back, so its next counter update and queue entries need no release.
                left = __hip_atomic_fetch_add(g.items_left + task, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - 1;
            }
            left = __builtin_amdgcn_readfirstlane(left);
            if (left == 0) {
                // last item of the task: release its successors, one per lane (a task of an n-tile column has up to n
                // of them; each costs two dependent memory round trips, its counter and its queue's tail).
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
                for (int q = tid; q < tc.edge_cnt; q += 64) {
                    if (q >= 64) ed = g.edges[tc.edge_off + q];
                    const int d =
                        __hip_atomic_fetch_add(g.deps + ed.succ, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - 1;
                    if (d == 0) {
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
                        push_task(g, ed);
                    }
                }
                if (tid == 0) __hip_atomic_fetch_add(g.done_items, tc.n_items, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            if (tid == 0) {
                if (g.trace) {  // {entry, workgroup, start, end, end of the successor release (last item only), 0}
                    const int slot =
                        __hip_atomic_fetch_add(g.trace_cursor, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (slot < g.total_items) {
                        uint64_t* rec = g.trace + TRACE_WORDS * (long)slot;
                        rec[0] = (uint64_t)e;
                        rec[1] = blockIdx.x;
                        rec[2] = t0;
                        rec[3] = t1;
                        rec[4] = left == 0 ? wall_clock64() : 0;
                        rec[5] = 0;
                    }
                }
                if (primary) __hip_atomic_fetch_add(idle_primary, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (tc.crit) __hip_atomic_fetch_add(g.cu_crit + my_key, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
}

// Restores the counters and queues of a graph, and clears the pivot reports, POTRF flags and locks of its matrices, so
// that it can run (again).
__global__ void k_graph_reset(DevGraph g, int n_slots) {
    const int stride = gridDim.x * blockDim.x;
    for (int x = blockIdx.x * blockDim.x + threadIdx.x; x < n_slots; x += stride) g.q_items[x] = g.q_items0[x];
    for (int x = blockIdx.x * blockDim.x + threadIdx.x; x < g.n_tasks; x += stride) {
        g.deps[x] = g.deps0[x];
        g.items_left[x] = g.tasks[x].n_items;
        const DevTask t = g.tasks[x];
        if (t.kind == K_GEMM || t.kind == K_SYRK) {
            const DevMat& M = g.mats[t.mat];
            const long nt = M.nt;
            for (int q = 0; q < t.kspan; q++) {
                GemmOperands o;
                o.A = M.tiles[t.i + (t.k + q) * nt];
                o.B = M.tiles[t.j + (t.k + q) * nt];
                o.C = M.tiles[t.i + t.j * nt];
                o.PA = M.planes ? M.planes[t.i + (t.k + q) * nt] : nullptr;
                o.PB = M.planes ? M.planes[t.j + (t.k + q) * nt] : nullptr;
                o.m = M.bsz[t.i];
                o.n = M.bsz[t.j];
                o.K = M.bsz[t.k + q];
                o.pad = 0;
                g.gops[(long)x * g.gop_stride + q] = o;
            }
        }
    }
    for (long x = blockIdx.x * blockDim.x + threadIdx.x; x < (long)g.n_tasks * NXCD; x += stride) g.xcd_run[x] = 0;
    for (int x = blockIdx.x * blockDim.x + threadIdx.x; x < g.n_buckets; x += stride) {
        g.q_head[x] = 0;
        g.q_tail[x] = g.tail0[x];
        g.q_count[x] = g.tail0[x];
    }
    for (int x = blockIdx.x * blockDim.x + threadIdx.x; x < CU_KEYS; x += stride) {
        g.cu_slots[x] = 0;
        g.cu_crit[x] = 0;
    }
    for (int x = blockIdx.x * blockDim.x + threadIdx.x; x < NXCD * 64; x += stride) g.idle_primary[x] = 0;
    for (int q = 0; q < g.n_bound; q++) {
        const DevMat& M = g.mats[g.bound[q]];
        for (int x = blockIdx.x * blockDim.x + threadIdx.x; x < M.nt * M.pf_stride; x += stride) M.pflags[x] = 0;
        if (g.has_accum)
            for (long x = blockIdx.x * blockDim.x + threadIdx.x; x < (long)M.nt * M.nt * 16; x += stride) M.locks[x] = 0;
        if (blockIdx.x == 0 && threadIdx.x == 0) *M.info = 0;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *g.done_items = 0;
        *g.abort_flag = 0;
        if (g.trace_cursor) *g.trace_cursor = 0;
    }
}
__global__ void k_graph_report(DevGraph g, GraphReport* out, int seq) {
    if (threadIdx.x != 0) return;
    int info = 0;
    for (int q = 0; q < g.n_bound && info == 0; q++) info = *g.mats[g.bound[q]].info;
    out->done = *g.done_items;
    out->abort_code = *g.abort_flag;
    out->info = info;
    __atomic_thread_fence(__ATOMIC_RELEASE);  // system scope
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __hip_atomic_store(&out->seq, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------------------------------------------------------------------
// Raw tile kernels behind the BLAS-shaped C-ABI entry points.
// ---------------------------------------------------------------------------
template <typename TS, int PREC, int BM>
__global__ __launch_bounds__(NTHREADS, 2) void k_raw_gemm(const TS* A, long lda, const TS* B, long ldb, TS* C, long ldc,
                                                          int m, int n, int K, int syrk, double alpha, double beta) {
    extern __shared__ __align__(16) char lds[];
    static_assert(2 * (gemm_item_lds<TS, PREC, BM>() + 1024) <= 160 * 1024, "two workgroups per CU");
    int rb, cb;
    decode_gemm_item(blockIdx.x, (m + BM - 1) / BM, syrk != 0, rb, cb);
    item_gemm<TS, PREC, BM>(A, lda, B, ldb, C, ldc, m, n, K, rb * BM, cb * BM, syrk != 0, alpha, beta, lds);
}

// The items wait only on lower-numbered blocks of the launch, which are dispatched first.
template <typename TS>
__global__ __launch_bounds__(NTHREADS, 2) void k_raw_potrf(TS* A, long lda, int n, double* dinv, int* info,
                                                           int32_t* flags, int32_t* err) {
    extern __shared__ __align__(16) char lds[];
    item_potrf<TS>(A, lda, n, dinv, info, 0, blockIdx.x, flags, err, (int64_t)500000000, lds);
}

// IN_LDS: the form that keeps the solved columns in LDS.
template <typename TS, bool IN_LDS> constexpr int raw_trsm_lds() {
    return IN_LDS ? trsm_lds_bytes<TS>() : sizeof(TS) == 8 ? LDS_TRSM : LDS_TRSM_F32;
}
template <typename TS, bool IN_LDS>
__global__ __launch_bounds__(NTHREADS, 2) void k_raw_trsm(const TS* L, long ldl, const double* dinv, TS* X, long ldx,
                                                          int m, int n) {
    extern __shared__ __align__(16) char lds[];
    const int r0 = blockIdx.x * trsm_rows(sizeof(TS), IN_LDS);
    if constexpr (IN_LDS) item_trsm_lds<TS>(L, ldl, dinv, X, ldx, m, n, r0, lds);
    else item_trsm<TS, TS>(L, ldl, dinv, X, ldx, m, n, r0, lds);
}

// Inverses of the 64x64 diagonal blocks of a lower-triangular n x n L (one block per workgroup).
template <typename TS>
__global__ __launch_bounds__(NTHREADS) void k_trtri_diag(const TS* L, long ldl, int n, double* dinv) {
    __shared__ double D[DB * DP];
    __shared__ double Xs[DB * DP];
    const int pb = blockIdx.x, p0 = pb * DB, pw = min(DB, n - p0);
    for (int e = threadIdx.x; e < DB * DB; e += NTHREADS) {
        const int i = e % DB, j = e / DB;
        D[i + j * DP] = (i < pw && j < pw && i >= j) ? (double)L[(p0 + i) + (long)(p0 + j) * ldl] : (i == j ? 1.0 : 0.0);
    }
    __syncthreads();
    lds_trtri64(D, Xs, pw);
    double* X = dinv + (long)pb * DB * DB;
    for (int e = threadIdx.x; e < DB * DB; e += NTHREADS) X[e] = Xs[(e % DB) + (e / DB) * DP];
}

// ---------------------------------------------------------------------------
// Tile layout conversion: full column-major n x n (FP64) <-> lower tiles. Workgroups (i, j, z) share tile (i, j): every
// gridDim.z-th group of CONV_COLS columns, a wave per column, each lane CONV_U accesses of V consecutive rows in flight: V = 2
// (16 bytes of FP64) where the dense array's alignment and the tile's rows allow it. Bound by HBM. (One workgroup per
// tile, an element at a time with a division each: n = 2048, b = 256 93 us to pack and 104 to unpack, now 10 and 10;
// n = 16384, b = 512 0.88 and 1.25 ms, now 0.51 and 0.65.)
// SMALL (no tile above CONV_SMALL rows): one workgroup per tile, element by element. A wave per column leaves lanes idle
// there, and what bounds it is the launch of the workgroups and what each does before its first access. FP64, us to pack and
// unpack with a wave per column / so: n = 4096, b = 8 127 and 230 / 72 and 98; n = 8192, b = 32 175 and 301 / 101 and 160,
// b = 64 127 and 201 / 115 and 174 (b = 128 126 and 170, so 150 and 224).
// ---------------------------------------------------------------------------
constexpr int CONV_COLS = 16, CONV_U = 4, CONV_SMALL = 64;
template <typename T, int V> struct ConvVec { typedef T t __attribute__((ext_vector_type(V))); };
template <typename T> struct ConvVec<T, 1> { typedef T t; };
// load(row, column) and store(row, column, value) for the first rows of every V-row access of this workgroup's groups of
// columns of an r x c tile, CONV_U at a time: load all, then store all.
template <int V, typename L, typename S>
__device__ __forceinline__ void conv_tile(int r, int c, const L& load, const S& store) {
    const int lane = threadIdx.x & 63;
    for (int g = blockIdx.z; g * CONV_COLS < c; g += gridDim.z) {
        const int q0 = g * CONV_COLS + (threadIdx.x >> 6), q1 = min(c, (g + 1) * CONV_COLS);
        for (int q = q0; q < q1; q += 4)
            for (int p0 = V * lane; p0 < r; p0 += 64 * V * CONV_U) {
                decltype(load(0, 0)) v[CONV_U];
#pragma unroll
                for (int u = 0; u < CONV_U; u++)
                    if (p0 + u * 64 * V < r) v[u] = load(p0 + u * 64 * V, q);
#pragma unroll
                for (int u = 0; u < CONV_U; u++)
                    if (p0 + u * 64 * V < r) store(p0 + u * 64 * V, q, v[u]);
            }
    }
}
// The same for a matrix of small tiles: the tile's elements one by one, over all threads.
template <typename L, typename S>
__device__ __forceinline__ void conv_small(int r, int c, const L& load, const S& store) {
    for (int e0 = threadIdx.x; e0 < r * c; e0 += NTHREADS * CONV_U) {
        decltype(load(0, 0)) v[CONV_U];
#pragma unroll
        for (int u = 0; u < CONV_U; u++) {
            const int e = e0 + u * NTHREADS;
            if (e < r * c) v[u] = load(e % r, e / r);
        }
#pragma unroll
        for (int u = 0; u < CONV_U; u++) {
            const int e = e0 + u * NTHREADS;
            if (e < r * c) store(e % r, e / r, v[u]);
        }
    }
}
// Two rows per access need 16-byte aligned pairs of the dense array and whole pairs in the tile's columns.
__device__ __forceinline__ bool conv_pairs(const double* dense, long ld, int r) {
    return ((uintptr_t)dense % 16) == 0 && (ld % 2) == 0 && (r % 2) == 0;
}

template <typename TS, bool SMALL>
__global__ __launch_bounds__(NTHREADS) void k_pack(const double* __restrict__ src, long lda, const DevMat* M, int nt) {
    const int i = blockIdx.x, j = blockIdx.y;
    if (i < j) return;
    const DevMat& m = *M;
    const int r = m.bsz[i], c = m.bsz[j];
    TTAD_GLOBAL TS* t = gmem((TS*)m.tiles[i + (long)j * nt]);
    const double* base = src + m.boff[i] + (long)m.boff[j] * lda;
    auto run = [&](auto vc) {
        constexpr int V = decltype(vc)::value;
        typedef typename ConvVec<double, V>::t sv;
        typedef typename ConvVec<TS, V>::t dv;
        auto load = [&](int p, int q) { return *reinterpret_cast<const TTAD_GLOBAL sv*>(gmem(base) + p + (long)q * lda); };
        auto store = [&](int p, int q, sv v) {
            if constexpr (V == 1) t[p + (long)q * r] = (TS)v;
            else *reinterpret_cast<TTAD_GLOBAL dv*>(t + p + (long)q * r) = __builtin_convertvector(v, dv);
        };
        if constexpr (SMALL) conv_small(r, c, load, store);
        else conv_tile<V>(r, c, load, store);
    };
    if constexpr (SMALL) run(std::integral_constant<int, 1>{});
    else if (conv_pairs(base, lda, r)) run(std::integral_constant<int, 2>{});
    else run(std::integral_constant<int, 1>{});
}
template <typename TS, bool SMALL>
__global__ __launch_bounds__(NTHREADS) void k_unpack(double* __restrict__ dst, long ldd, const DevMat* M, int nt, int zero_upper) {
    const int i = blockIdx.x, j = blockIdx.y;
    if (i < j && !zero_upper) return;
    const DevMat& m = *M;
    const int r = m.bsz[i], c = m.bsz[j];
    const TTAD_GLOBAL TS* t = i < j ? nullptr : gmem((const TS*)m.tiles[i + (long)j * nt]);
    double* base = dst + m.boff[i] + (long)m.boff[j] * ldd;
    auto run = [&](auto vc) {
        constexpr int V = decltype(vc)::value;
        typedef typename ConvVec<double, V>::t dv;
        typedef typename ConvVec<TS, V>::t sv;
        auto load = [&](int p, int q) {
            if (i < j) return dv(0);
            if constexpr (V == 1) return (double)t[p + (long)q * r];
            else return __builtin_convertvector(*reinterpret_cast<const TTAD_GLOBAL sv*>(t + p + (long)q * r), dv);
        };
        auto store = [&](int p, int q, dv v) {
            TTAD_GLOBAL double* d = gmem(base) + p + (long)q * ldd;
            if (i == j && p < q) {  // the strict upper triangle
                if constexpr (V == 1) {
                    if (zero_upper) *d = 0.0;
                } else {
                    if (p + 1 < q) v[1] = 0.0;
                    v[0] = 0.0;
                    if (zero_upper) *reinterpret_cast<TTAD_GLOBAL dv*>(d) = v;
                    else if (p + 1 >= q) d[1] = v[1];
                }
                return;
            }
            *reinterpret_cast<TTAD_GLOBAL dv*>(d) = v;
        };
        if constexpr (SMALL) conv_small(r, c, load, store);
        else conv_tile<V>(r, c, load, store);
    };
    if constexpr (SMALL) run(std::integral_constant<int, 1>{});
    else if (conv_pairs(base, ldd, r)) run(std::integral_constant<int, 2>{});
    else run(std::integral_constant<int, 1>{});
}
// Tile-wise copy with conversion between two matrices of the same partition, one workgroup of 256 per lower
// tile (workgroup x -> tile (i, j), x = i (i + 1) / 2 + j). Four consecutive elements move as one vector access
// (two 16-byte loads of FP64, one 16-byte store of FP32), four quads in flight per thread; a tile whose pointers
// or element count do not allow quads is copied element by element.
template <typename TD, typename TSRC>
__global__ __launch_bounds__(256) void k_copy_tiles(const DevMat* S, const DevMat* D, int nt) {
    typedef TSRC s4 __attribute__((ext_vector_type(4)));
    typedef TD d4 __attribute__((ext_vector_type(4)));
    const int x = blockIdx.x;
    int i = (int)((sqrt(8.0 * x + 1.0) - 1.0) * 0.5);
    while ((i + 1) * (i + 2) / 2 <= x) i++;
    while (i * (i + 1) / 2 > x) i--;
    const int j = x - i * (i + 1) / 2;
    const TSRC* s = (const TSRC*)S->tiles[i + (long)j * nt];
    TD* d = (TD*)D->tiles[i + (long)j * nt];
    const long cnt = (long)S->bsz[i] * S->bsz[j];
    const bool quads = (cnt % 4) == 0 && ((uintptr_t)s % sizeof(s4)) == 0 && ((uintptr_t)d % sizeof(d4)) == 0;
    if (!quads) {
        for (long e = threadIdx.x; e < cnt; e += 256) d[e] = (TD)s[e];
        return;
    }
    const TTAD_GLOBAL s4* sp = gmem((const s4*)s);
    TTAD_GLOBAL d4* dp = gmem((d4*)d);
    const long nq = cnt / 4;
    long e = threadIdx.x;
    for (; e + 3 * 256 < nq; e += 4 * 256) {
        const s4 v0 = sp[e], v1 = sp[e + 256], v2 = sp[e + 512], v3 = sp[e + 768];
        dp[e] = __builtin_convertvector(v0, d4);
        dp[e + 256] = __builtin_convertvector(v1, d4);
        dp[e + 512] = __builtin_convertvector(v2, d4);
        dp[e + 768] = __builtin_convertvector(v3, d4);
    }
    for (; e < nq; e += 256) dp[e] = __builtin_convertvector(sp[e], d4);
}

// ---------------------------------------------------------------------------
// Launch wrappers (host side, C++ linkage; called by the C-ABI layer).
// ---------------------------------------------------------------------------
static hipError_t set_lds(const void* f, int bytes) {
    return hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

hipError_t kernels_init() {
    hipError_t e = hipSuccess;
#define TTAD_SETLDS2(fn, bytes)                      \
    do {                                             \
        e = set_lds((const void*)(fn), (bytes));     \
        if (e != hipSuccess) return e;               \
    } while (0)
    TTAD_SETLDS2(k_items<VSETS[0]>, vset_lds(VSETS[0]));
    TTAD_SETLDS2(k_items<VSETS[1]>, vset_lds(VSETS[1]));
    TTAD_SETLDS2(k_items<VSETS[2]>, vset_lds(VSETS[2]));
    TTAD_SETLDS2(k_items<VSETS[3]>, vset_lds(VSETS[3]));
    TTAD_SETLDS2(k_items<VSETS[4]>, vset_lds(VSETS[4]));
    TTAD_SETLDS2(k_items<VSETS[5]>, vset_lds(VSETS[5]));
    TTAD_SETLDS2(k_persistent<VSETS[0]>, vset_lds(VSETS[0]));
    TTAD_SETLDS2(k_persistent<VSETS[1]>, vset_lds(VSETS[1]));
    TTAD_SETLDS2(k_persistent<VSETS[2]>, vset_lds(VSETS[2]));
    TTAD_SETLDS2(k_persistent<VSETS[3]>, vset_lds(VSETS[3]));
    TTAD_SETLDS2(k_persistent<VSETS[4]>, vset_lds(VSETS[4]));
    TTAD_SETLDS2(k_persistent<VSETS[5]>, vset_lds(VSETS[5]));
    TTAD_SETLDS2(k_persistent<VSETS[6]>, vset_lds(VSETS[6]));
#define TTAD_SETLDS_GEMM(ts, prec)                                                                        \
    TTAD_SETLDS2((k_raw_gemm<ts, prec, GEMM_BM>), (gemm_item_lds<ts, prec, GEMM_BM>()));                   \
    TTAD_SETLDS2((k_raw_gemm<ts, prec, GEMM_BS>), (gemm_item_lds<ts, prec, GEMM_BS>()))
    TTAD_SETLDS_GEMM(double, P_F64);
    TTAD_SETLDS_GEMM(float, P_F32);
    TTAD_SETLDS_GEMM(float, P_BF16);
    TTAD_SETLDS_GEMM(float, P_BF16X3);
#undef TTAD_SETLDS_GEMM
    TTAD_SETLDS2((k_raw_potrf<double>), LDS_POTRF);
    TTAD_SETLDS2((k_raw_potrf<float>), LDS_POTRF);
    TTAD_SETLDS2((k_raw_trsm<double, true>), (raw_trsm_lds<double, true>()));
    TTAD_SETLDS2((k_raw_trsm<double, false>), (raw_trsm_lds<double, false>()));
    TTAD_SETLDS2((k_raw_trsm<float, true>), (raw_trsm_lds<float, true>()));
    TTAD_SETLDS2((k_raw_trsm<float, false>), (raw_trsm_lds<float, false>()));
#undef TTAD_SETLDS2
    return e;
}

static const void* persistent_fn(int vset) {
    switch (vset) {
        case 0: return (const void*)k_persistent<VSETS[0]>;
        case 1: return (const void*)k_persistent<VSETS[1]>;
        case 2: return (const void*)k_persistent<VSETS[2]>;
        case 3: return (const void*)k_persistent<VSETS[3]>;
        case 4: return (const void*)k_persistent<VSETS[4]>;
        case 5: return (const void*)k_persistent<VSETS[5]>;
        default: return (const void*)k_persistent<VSETS[6]>;
    }
}

static int vset_lds_of(int vset) {
    switch (vset) {
        case 0: return vset_lds(VSETS[0]);
        case 1: return vset_lds(VSETS[1]);
        case 2: return vset_lds(VSETS[2]);
        case 3: return vset_lds(VSETS[3]);
        case 4: return vset_lds(VSETS[4]);
        case 5: return vset_lds(VSETS[5]);
        default: return vset_lds(VSETS[6]);
    }
}

int persistent_blocks_per_cu(int vset) {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, persistent_fn(vset), NTHREADS, vset_lds_of(vset)) !=
        hipSuccess)
        return 1;
    return nb > 0 ? nb : 1;
}

void launch_items(int vset, const DevMat* mats, const DevTask* tasks, const int32_t* prefix, int n_tasks,
                  int n_items, int32_t* err, hipStream_t s) {
    if (n_items <= 0) return;
    const dim3 grid(n_items), block(NTHREADS);
    // (no accumulate-mode variant here: host-sequenced plans hold no accumulate tasks)
    const int lds = vset_lds_of(std::min(vset, N_VSETS - 2));
    switch (vset) {
        case 0: hipLaunchKernelGGL(k_items<VSETS[0]>, grid, block, lds, s, mats, tasks, prefix, n_tasks, err); break;
        case 1: hipLaunchKernelGGL(k_items<VSETS[1]>, grid, block, lds, s, mats, tasks, prefix, n_tasks, err); break;
        case 2: hipLaunchKernelGGL(k_items<VSETS[2]>, grid, block, lds, s, mats, tasks, prefix, n_tasks, err); break;
        case 3: hipLaunchKernelGGL(k_items<VSETS[3]>, grid, block, lds, s, mats, tasks, prefix, n_tasks, err); break;
        case 4: hipLaunchKernelGGL(k_items<VSETS[4]>, grid, block, lds, s, mats, tasks, prefix, n_tasks, err); break;
        default: hipLaunchKernelGGL(k_items<VSETS[5]>, grid, block, lds, s, mats, tasks, prefix, n_tasks, err); break;
    }
}

__global__ void k_read_clock(uint64_t* out) {
    if (threadIdx.x == 0) *out = wall_clock64();
}
void launch_read_clock(uint64_t* out, hipStream_t s) { hipLaunchKernelGGL(k_read_clock, dim3(1), dim3(64), 0, s, out); }

void launch_graph_reset(const DevGraph& g, int n_slots, hipStream_t s) {
    hipLaunchKernelGGL(k_graph_reset, dim3(256), dim3(256), 0, s, g, n_slots);
}
void launch_graph_report(const DevGraph& g, GraphReport* out, int seq, hipStream_t s) {
    hipLaunchKernelGGL(k_graph_report, dim3(1), dim3(64), 0, s, g, out, seq);
}

void launch_persistent(int vset, const DevGraph& g, int n_workers, hipStream_t s) {
    const dim3 grid(n_workers), block(NTHREADS);
    const int lds = vset_lds_of(vset);
    switch (vset) {
        case 0: hipLaunchKernelGGL(k_persistent<VSETS[0]>, grid, block, lds, s, g); break;
        case 1: hipLaunchKernelGGL(k_persistent<VSETS[1]>, grid, block, lds, s, g); break;
        case 2: hipLaunchKernelGGL(k_persistent<VSETS[2]>, grid, block, lds, s, g); break;
        case 3: hipLaunchKernelGGL(k_persistent<VSETS[3]>, grid, block, lds, s, g); break;
        case 4: hipLaunchKernelGGL(k_persistent<VSETS[4]>, grid, block, lds, s, g); break;
        case 5: hipLaunchKernelGGL(k_persistent<VSETS[5]>, grid, block, lds, s, g); break;
        default: hipLaunchKernelGGL(k_persistent<VSETS[6]>, grid, block, lds, s, g); break;
    }
}

template <typename TS, int PREC, int BM>
static void raw_gemm(const void* A, long lda, const void* B, long ldb, void* C, long ldc, int m, int n, int K, int syrk,
                     double alpha, double beta, hipStream_t s) {
    hipLaunchKernelGGL((k_raw_gemm<TS, PREC, BM>), dim3((unsigned)raw_gemm_items(m, n, syrk != 0, BM)), dim3(NTHREADS), (gemm_item_lds<TS, PREC, BM>()), s,
                       (const TS*)A, lda, (const TS*)B, ldb, (TS*)C, ldc, m, n, K, syrk, alpha, beta);
}

void launch_raw_gemm(int prec, const void* A, long lda, const void* B, long ldb, void* C, long ldc, int m, int n,
                     int K, int syrk, double alpha, double beta, hipStream_t s) {
    if (m <= 0 || n <= 0) return;
    const bool small = raw_gemm_small(prec, m, n, K, syrk != 0);
    auto* f = prec == P_F64    ? (small ? raw_gemm<double, P_F64, GEMM_BS> : raw_gemm<double, P_F64, GEMM_BM>)
              : prec == P_F32  ? (small ? raw_gemm<float, P_F32, GEMM_BS> : raw_gemm<float, P_F32, GEMM_BM>)
              : prec == P_BF16 ? (small ? raw_gemm<float, P_BF16, GEMM_BS> : raw_gemm<float, P_BF16, GEMM_BM>)
                               : (small ? raw_gemm<float, P_BF16X3, GEMM_BS> : raw_gemm<float, P_BF16X3, GEMM_BM>);
    f(A, lda, B, ldb, C, ldc, m, n, K, syrk, alpha, beta, s);
}

void launch_raw_potrf(int prec, void* A, long lda, int n, double* dinv, int* info, int32_t* flags, int32_t* err,
                      hipStream_t s) {
    const dim3 grid(potrf_items(n)), block(NTHREADS);
    if (prec == P_F64)
        hipLaunchKernelGGL((k_raw_potrf<double>), grid, block, LDS_POTRF, s, (double*)A, lda, n, dinv, info, flags, err);
    else
        hipLaunchKernelGGL((k_raw_potrf<float>), grid, block, LDS_POTRF, s, (float*)A, lda, n, dinv, info, flags, err);
}

void launch_trtri_diag(int prec, const void* L, long ldl, int n, double* dinv, hipStream_t s) {
    const int nb = (n + DB - 1) / DB;
    if (prec == P_F64)
        hipLaunchKernelGGL((k_trtri_diag<double>), dim3(nb), dim3(NTHREADS), 0, s, (const double*)L, ldl, n, dinv);
    else
        hipLaunchKernelGGL((k_trtri_diag<float>), dim3(nb), dim3(NTHREADS), 0, s, (const float*)L, ldl, n, dinv);
}

template <typename TS, bool IN_LDS>
static void raw_trsm(const void* L, long ldl, const double* dinv, void* X, long ldx, int m, int n, hipStream_t s) {
    const int bm = trsm_rows(sizeof(TS), IN_LDS);
    hipLaunchKernelGGL((k_raw_trsm<TS, IN_LDS>), dim3((m + bm - 1) / bm), dim3(NTHREADS),
                       (raw_trsm_lds<TS, IN_LDS>()), s, (const TS*)L, ldl, dinv, (TS*)X, ldx, m, n);
}

void launch_raw_trsm(int prec, const void* L, long ldl, const double* dinv, void* X, long ldx, int m, int n,
                     hipStream_t s) {
    if (m <= 0) return;
    const bool in_lds = ldl < TRSM_LDS_MAX_LD && ldx < TRSM_LDS_MAX_LD && trsm_in_lds(prec == P_F64 ? 8 : 4, m, n);
    auto* f = prec == P_F64 ? (in_lds ? raw_trsm<double, true> : raw_trsm<double, false>)
                            : (in_lds ? raw_trsm<float, true> : raw_trsm<float, false>);
    f(L, ldl, dinv, X, ldx, m, n, s);
}

// Workgroups per tile: one per group of the largest tile's columns, but no more than 2^20 in all where tiles are many (a
// partition of small tiles and a few large ones would launch mostly empty ones: 512 tiles of 16 and one of 2048, 7.4 ms to pack
// and 9.2 to unpack, so 0.86 and 1.7).
static dim3 conv_grid(int nt, int max_b) {
    const long groups = max_b <= CONV_SMALL ? 1 : (max_b + CONV_COLS - 1) / CONV_COLS;
    return dim3(nt, nt, (unsigned)std::max(1L, std::min(groups, (1L << 20) / ((long)nt * nt))));
}

void launch_pack(int storage, const double* src, long lda, const DevMat* M, int nt, int max_b, hipStream_t s) {
    const bool small = max_b <= CONV_SMALL;
    auto* f = storage == P_F64 ? (small ? k_pack<double, true> : k_pack<double, false>)
                               : (small ? k_pack<float, true> : k_pack<float, false>);
    hipLaunchKernelGGL(f, conv_grid(nt, max_b), dim3(NTHREADS), 0, s, src, lda, M, nt);
}

void launch_unpack(int storage, double* dst, long ldd, const DevMat* M, int nt, int max_b, int zero_upper, hipStream_t s) {
    const bool small = max_b <= CONV_SMALL;
    auto* f = storage == P_F64 ? (small ? k_unpack<double, true> : k_unpack<double, false>)
                               : (small ? k_unpack<float, true> : k_unpack<float, false>);
    hipLaunchKernelGGL(f, conv_grid(nt, max_b), dim3(NTHREADS), 0, s, dst, ldd, M, nt, zero_upper);
}

void launch_copy_tiles(int dst_storage, int src_storage, const DevMat* S, const DevMat* D, int nt, hipStream_t s) {
    const unsigned nlow = (unsigned)nt * (nt + 1) / 2;
    if (dst_storage == P_F32 && src_storage == P_F64)
        hipLaunchKernelGGL((k_copy_tiles<float, double>), dim3(nlow), dim3(256), 0, s, S, D, nt);
    else if (dst_storage == P_F64 && src_storage == P_F32)
        hipLaunchKernelGGL((k_copy_tiles<double, float>), dim3(nlow), dim3(256), 0, s, S, D, nt);
    else if (dst_storage == P_F64)
        hipLaunchKernelGGL((k_copy_tiles<double, double>), dim3(nlow), dim3(256), 0, s, S, D, nt);
    else hipLaunchKernelGGL((k_copy_tiles<float, float>), dim3(nlow), dim3(256), 0, s, S, D, nt);
}

}  // namespace ttad
