// Device-side task execution: item dispatch, the host-sequenced item kernel and
// the persistent DAG kernel that replaces the Threadpool worker loop
// (tasktorrent/src/threadpool_shared.cpp:104-195) and the per-thread dependency
// maps of Taskflow::fulfill_promise (tasktorrent/src/taskflow.hpp:241-296).
#pragma once
#include "tile_ops.hpp"

namespace ttad {

// Device image of a task graph (built on the host from the Taskflow callbacks).
struct DevGraph {
    int32_t n_tasks;
    int32_t n_buckets;
    int32_t total_items;
    const DevTask* tasks;
    const DevEdge* edges;       // out-edges, by task
    const int32_t* deps0;       // initial dependency counters (indegree - host seeds)
    const int32_t* tail0;       // initial queue tails per bucket
    const int64_t* q_items0;    // [total_items] initial queue entries: those of ready tasks, else -1
    int32_t n_bound;
    const int32_t* bound;       // [n_bound] the slots of mats that a matrix is bound to
    int32_t has_accum;          // some update runs in accumulate mode (the tile locks are cleared before a run)
    int32_t* deps;
    int32_t* items_left;
    int32_t* q_head;            // [n_buckets]
    int32_t* q_tail;            // [n_buckets]
    int32_t* q_count;           // [n_buckets] entries pushed and not yet claimed (dips below zero while
                                // a failed claim gives its credit back)
    const int32_t* q_base;      // [n_buckets+1]
    const int32_t* q_home;      // [n_buckets] -1 = any worker, else the XCD served first
    int64_t* q_items;           // entries (task << 20) | item; -1 = not yet written
    int32_t* done_items;
    int32_t* abort_flag;        // 1 = watchdog, 2 = queue overflow
    const DevMat* mats;
    GemmOperands* gops;         // [n_tasks * gop_stride] resolved operands of the GEMM/SYRK tasks' steps (filled before
                                // each run)
    int32_t gop_stride;         // the largest kspan
    uint64_t* trace;            // optional: TRACE_WORDS x u64 per item {task<<20|item, wg, t_start, t_end,
                                // t_end of the successor release (the task's last item; else 0), 0}
    int32_t* trace_cursor;
    int32_t* cu_slots;          // [CU_KEYS] workers started per CU (slot 0 = primary)
    int32_t* idle_primary;      // [NXCD * 64] primary workers currently looking for work, per XCD (entry 64 * x)
    int32_t* cu_crit;           // [CU_KEYS] critical items running per CU (its other worker waits)
    int32_t* xcd_run;           // [n_tasks * NXCD] items of a task running on each XCD (release elision)
    int64_t spin_limit;         // watchdog in wall_clock64 ticks
};

constexpr int TRACE_WORDS = 6;  // u64 per trace record

// What a finished run tells the host, in pinned memory; seq is written last.
struct GraphReport {
    int32_t done, abort_code;
    int32_t info;  // of the first bound matrix with a non-positive pivot, else 0
    int32_t seq;
};

// XCDs of the device (MI355X: 8 XCDs of 32 CUs, each with its own L2).
constexpr int NXCD = 8;
// Work queues of a graph: 64 priority buckets, each with a shared queue and one queue homed on each
// XCD. Bucket b's shared queue is queue b * QUEUE_SHARED_STRIDE (every worker claims from the shared
// queues: their counters get a cache line each), its queue homed on XCD x is
// QUEUE_HOMED + x * QUEUE_BUCKETS + b (only that XCD's workers and stealers claim there: the 64 counters
// of one XCD share 256 bytes and no line with another XCD's). The ids in between are empty queues.
// A scan reads one bucket per lane of a wave.
constexpr int QUEUE_BUCKETS = 64;
constexpr int QUEUE_SHARED_STRIDE = 32;  // 128-byte lines of 4-byte counters
constexpr int QUEUE_HOMED = QUEUE_BUCKETS * QUEUE_SHARED_STRIDE;
constexpr int MAX_QUEUES = QUEUE_HOMED + QUEUE_BUCKETS * NXCD;
__host__ __device__ constexpr int shared_queue(int b) { return b * QUEUE_SHARED_STRIDE; }
__host__ __device__ constexpr int homed_queue(int x, int b) { return QUEUE_HOMED + x * QUEUE_BUCKETS + b; }
constexpr int CLAIM_TRIES = 4;  // queues a claimer tries from one scan
constexpr int IDLE_PRIMARIES = 8;  // idle primaries of an XCD (32 CUs) from which on its secondaries hold back
constexpr int IDLE_BACKOFF = 10;  // log2 of the longest pause between the looks of an idle worker, x 64 cycles
// Hardware id of the XCD (XCC) this wave runs on.
__device__ __forceinline__ int xcc_id() {
    unsigned v;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(v));
    return (int)(v & 0xF) % NXCD;
}

// Identifier of the CU this wave runs on: XCC, shader engine, shader array and CU fields of
// the hardware id registers (fewer than CU_KEYS values).
constexpr int CU_KEYS = 2048;
__device__ __forceinline__ int cu_key() {
    unsigned hw;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_HW_ID)" : "=s"(hw));
    const int cu = (hw >> 8) & 15, sh = (hw >> 12) & 1, se = (hw >> 13) & 7;
    return ((xcc_id() * 8 + se) * 2 + sh) * 16 + cu;
}

__device__ __forceinline__ int ld_relaxed(const int32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int64_t ld_acquire64(const int64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int64_t ld_relaxed64(const int64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Item variants a kernel is compiled with (bit mask). A kernel holding every
// variant allocates registers for the largest one; the executors are therefore
// instantiated per precision and the host picks the smallest set that covers a graph.
enum ItemVariant : int {
    V_F64S = 1,      // FP64 tiles: POTRF, TRSM, GEMM/SYRK on FP64 MFMA
    V_F32S = 2,      // FP32 tiles: POTRF (FP64 arithmetic), TRSM on FP32 MFMA
    V_G32 = 4,       // GEMM/SYRK FP32
    V_GBF16 = 8,     // GEMM/SYRK BF16
    V_GBF16X3 = 16,  // GEMM/SYRK BF16x3
    V_TLDS = 64,     // TRSM with the solved columns in LDS
    V_ACC = 32       // accumulate-mode GEMM/SYRK (only in the last set, so the others keep their registers)
};
// The compiled sets, smallest first.
// (FP64 tiles have two: large factorizations bound by the updates run the one without the TRSM form in LDS. n = 16384 alike,
// 25.7 ms; n = 24576 80.0 ms, 80.5 with the other set, 80.9 with its TRSM form too; n = 32768 185.0, 186.0 and 187.0.)
constexpr int V_ALL = V_F64S | V_F32S | V_G32 | V_GBF16 | V_GBF16X3 | V_TLDS;
constexpr int N_VSETS = 7;
constexpr int VSETS[N_VSETS] = {V_F64S, V_F64S | V_TLDS, V_F32S | V_G32 | V_TLDS, V_F32S | V_GBF16 | V_TLDS,
                                V_F32S | V_GBF16X3 | V_TLDS, V_ALL, V_ALL | V_ACC};

__host__ __device__ inline int item_variant(int kind, int prec, int storage) {
    if (kind == K_GEMM || kind == K_SYRK)
        return prec == P_F64 ? V_F64S : prec == P_F32 ? V_G32 : prec == P_BF16 ? V_GBF16 : V_GBF16X3;
    return storage == P_F64 ? V_F64S : V_F32S;
}
// LDS of an executor instantiation: the largest item of its variants.
constexpr int vset_lds(int vm) {
    int b = 0;
    if (vm & V_F64S) b = cmax(b, cmax(cmax(LDS_GEMM_F64, LDS_POTRF), LDS_TRSM));
    if (vm & V_F64S) b = cmax(b, gemm_item_lds<double, P_F64, GEMM_BS>());
    if (vm & V_G32) b = cmax(b, gemm_item_lds<float, P_F32, GEMM_BS>());
    if ((vm & V_TLDS) && (vm & V_F64S)) b = cmax(b, trsm_lds_bytes<double>());
    if ((vm & V_TLDS) && (vm & V_F32S)) b = cmax(b, trsm_lds_bytes<float>());
    if (vm & V_F32S) b = cmax(b, cmax(LDS_POTRF, LDS_TRSM_F32));
    if (vm & V_G32) b = cmax(b, LDS_GEMM_F32);
    if (vm & V_GBF16) b = cmax(b, LDS_GEMM_BF16_1);
    if (vm & V_GBF16X3) b = cmax(b, LDS_GEMM_BF16);
    return b;
}
// Workgroups per CU an instantiation is compiled for: two when two of them fit the CU's
// 160 KB of LDS (registers are then capped at 256 per lane, VGPRs and AGPRs together).
constexpr int vset_occupancy(int vm) { return 2 * (vset_lds(vm) + 1024) <= 160 * 1024 ? 2 : 1; }
inline int vset_index(int needed) {
    for (int q = 0; q < N_VSETS; q++)
        if ((needed & ~VSETS[q]) == 0) return q;
    return N_VSETS - 1;
}

// POTRF and TRSM items are called out of line from the executors: a kernel holding them
// inline is register-allocated for their largest live set and spills in the GEMM loop,
// which runs far more often. The call saves the callee's registers once per item.
// Their arguments arrive in vector registers; they are moved to scalar ones, so that sizes, addresses and the
// branches on them are scalar.
// One instance per executor instantiation (VM): a callee shared by kernels compiled for
// different occupancies would be register-allocated for the lowest of them.
// POTRF and TRSM carry the critical path: their waves run at raised issue priority, so
// that a GEMM item sharing the CU (two workgroups per CU) does not halve their MFMA share.
template <typename TS, int VM>
__device__ __attribute__((noinline)) void potrf_call(TS* A, long lda, int n, double* dinv, int* info, int col_off,
                                                     int it, int32_t* flags, int32_t* err, int64_t spin_limit,
                                                     char* lds) {
    __builtin_amdgcn_s_setprio(3);
    item_potrf<TS>(wave_uniform(A), wave_uniform((int)lda), wave_uniform(n), wave_uniform(dinv), wave_uniform(info),
                   wave_uniform(col_off), wave_uniform(it), wave_uniform(flags), wave_uniform(err), spin_limit,
                   lds_uniform(lds));
    __builtin_amdgcn_s_setprio(0);
}
// Accumulate-mode GEMM items are called out of line too, so the default GEMM loop keeps its registers.
template <typename TS, int PREC, int VM>
__device__ __attribute__((noinline)) void gemm_acc_call(const TS* A, long lda, const TS* B, long ldb, TS* C, long ldc,
                                                        int m, int n, int K, int r0, int c0, bool syrk, int32_t* lock,
                                                        int32_t* err, int64_t spin_limit, char* lds) {
    item_gemm_acc<TS, PREC>(A, lda, B, ldb, C, ldc, m, n, K, r0, c0, syrk, -1.0, lock, err, spin_limit, lds);
}
// 64x64 GEMM/SYRK items, out of line for the same reason. They are few and on or near the critical path, so their
// waves run at raised priority like POTRF's and TRSM's.
template <typename TS, int PREC, int VM>
__device__ __attribute__((noinline)) void gemm_small_call(const TS* A, const TS* B, TS* C, int m, int n, int K, int r0,
                                                          int c0, bool syrk, char* lds, const void* PA,
                                                          const void* PB) {
    __builtin_amdgcn_s_setprio(3);
    const int mu = wave_uniform(m), nu = wave_uniform(n);
    item_gemm<TS, PREC, GEMM_BS>(wave_uniform(A), mu, wave_uniform(B), nu, wave_uniform(C), mu, mu, nu, wave_uniform(K),
                                 wave_uniform(r0), wave_uniform(c0), wave_uniform((int)syrk) != 0, -1.0, 1.0,
                                 lds_uniform(lds), wave_uniform(PA), wave_uniform(PB));
    __builtin_amdgcn_s_setprio(0);
}
// The executor's 128x128 GEMM/SYRK items, `span` steps of K columns each with operands go[0 .. span - 1]: out of line, with
// registers of their own. Inline, the bf16x3 loop spilled with more than one step, and the FP64 loop's speed changed with
// whatever else the kernel held (n = 8192, b = 512, no fused task: 5.3 ms inline, 5.1 so). FOLD as item_gemm (with it the
// bf16x3 loop spills: n = 32768 45 -> 123 ms).
template <typename TS, int PREC, int VM, bool FOLD>
__device__ __attribute__((noinline)) void gemm_call(const GemmOperands* go, int span, int r0, int c0, bool syrk,
                                                    char* lds) {
    const GemmOperands* o = wave_uniform(go);
    const int m = wave_uniform(o->m), n = wave_uniform(o->n);
    item_gemm<TS, PREC, GEMM_BM, FOLD>((const TS*)wave_uniform(o->A), m, (const TS*)wave_uniform(o->B), n,
                                       (TS*)wave_uniform(o->C), m, m, n, wave_uniform(o->K), wave_uniform(r0),
                                       wave_uniform(c0), wave_uniform((int)syrk) != 0, -1.0, 1.0, lds_uniform(lds),
                                       wave_uniform(o->PA), wave_uniform(o->PB), o + 1, wave_uniform(span) - 1);
}
// LDS_FORM: the item may be one that keeps X in LDS (in_lds).
template <typename TS, int VM, bool LDS_FORM>
__device__ __attribute__((noinline)) void trsm_call(const TS* L, const double* dinv, TS* X, int m, int n, int it,
                                                    bool in_lds, char* lds, void* planes) {
    __builtin_amdgcn_s_setprio(3);
    const int mu = wave_uniform(m), nu = wave_uniform(n), iu = wave_uniform(it);
    char* l = lds_uniform(lds);
    bool done = false;
    if constexpr (LDS_FORM)
        if (wave_uniform((int)in_lds)) {
            item_trsm_lds<TS>(wave_uniform(L), nu, wave_uniform(dinv), wave_uniform(X), mu, mu, nu,
                              iu * trsm_rows(sizeof(TS), true), l, wave_uniform(planes));
            done = true;
        }
    if (!done)
        item_trsm<TS, TS>(wave_uniform(L), nu, wave_uniform(dinv), wave_uniform(X), mu, mu, nu,
                          iu * trsm_rows(sizeof(TS), false), l, wave_uniform(planes));
    __builtin_amdgcn_s_setprio(0);
}

// Execute work item `it` of task t. All 256 threads participate. Returns false
// (doing nothing) for an item variant outside VM. The items of a POTRF task wait on
// each other (item_potrf): the caller must
// have every lower-numbered item of the task running or done; their waits give up
// after spin_limit ticks or once *err is nonzero (and set *err = 1 when they time out).
// GOPS: the persistent executor's items, whose GEMM operands are resolved (go) and whose form t.sub chooses. Without, items
// are 128x128 and TRSM strips the higher ones (the host-sequenced schedule and the serving loop never ask for others).
template <int VM, bool GOPS = false>
__device__ __forceinline__ bool exec_item(const DevTask& t, int it, const DevMat* mats, char* lds, int32_t* err,
                                          int64_t spin_limit, const GemmOperands* go = nullptr) {
    if (t.kind == K_NOP) {  // spin task (scheduler-overhead benchmark): k device clock ticks, no tile access
        if (threadIdx.x == 0) {
            const uint64_t t0 = wall_clock64();
            while (wall_clock64() - t0 < (uint64_t)t.k) __builtin_amdgcn_s_sleep(1);
        }
        __syncthreads();
        return true;
    }
    const DevMat& M = mats[t.mat];
    const int nt = M.nt;
    auto tile = [&](int i, int j) { return M.tiles[i + (long)j * nt]; };
    auto planes = [&](int i, int j) { return M.planes ? M.planes[i + (long)j * nt] : nullptr; };
    const bool f64s = M.storage == P_F64;
    switch (t.kind) {
        case K_POTRF: {
            const int j = t.j, n = M.bsz[j];
            int32_t* flags = M.pflags + (long)j * M.pf_stride;
            if constexpr ((VM & V_F64S) != 0)
                if (f64s) {
                    potrf_call<double, VM>((double*)tile(j, j), n, n, M.dinv[j], M.info, M.boff[j], it, flags, err,
                                           spin_limit, lds);
                    return true;
                }
            if constexpr ((VM & V_F32S) != 0)
                if (!f64s) {
                    potrf_call<float, VM>((float*)tile(j, j), n, n, M.dinv[j], M.info, M.boff[j], it, flags, err,
                                          spin_limit, lds);
                    return true;
                }
            return false;
        }
        case K_TRSM: {
            const int i = t.i, j = t.j, m = M.bsz[i], n = M.bsz[j];
            const bool in_lds = t.sub == GEMM_BS;
            constexpr bool lds_form = GOPS && (VM & V_TLDS) != 0;
            if (!lds_form && in_lds) return false;
            if constexpr ((VM & V_F64S) != 0)
                if (f64s) {
                    trsm_call<double, VM, lds_form>((const double*)tile(j, j), M.dinv[j], (double*)tile(i, j), m, n, it, in_lds, lds,
                                        nullptr);
                    return true;
                }
            if constexpr ((VM & V_F32S) != 0)
                if (!f64s) {
                    trsm_call<float, VM, lds_form>((const float*)tile(j, j), M.dinv[j], (float*)tile(i, j), m, n, it, in_lds, lds,
                                        planes(i, j));
                    return true;
                }
            return false;
        }
        case K_SYRK:
        case K_GEMM: {
            const int k = t.k, i = t.i, j = t.j;
            const bool syrk = (t.kind == K_SYRK);
            const void *opA, *opB, *opPA, *opPB;
            void* opC;
            int m, n, K;
            // resolved before the run (persistent executor); the FP64 instantiation keeps the table lookups,
            // measured faster there (the FP64 items are long, the lookup latency is a small part of them)
            constexpr bool use_go = (VM & (V_G32 | V_GBF16 | V_GBF16X3)) != 0;
            const int span = wave_uniform(t.kspan);
            if (use_go && go) {
                opA = wave_uniform(go->A);
                opB = wave_uniform(go->B);
                opC = wave_uniform(go->C);
                opPA = wave_uniform(go->PA);
                opPB = wave_uniform(go->PB);
                m = wave_uniform(go->m);
                n = wave_uniform(go->n);
                K = wave_uniform(go->K);
            } else {
                opA = tile(i, k);
                opB = tile(j, k);
                opC = tile(i, j);
                opPA = planes(i, k);
                opPB = planes(j, k);
                m = M.bsz[i];
                n = M.bsz[j];
                K = M.bsz[k];
            }
            int rb, cb;
            const int sub = GOPS ? wave_uniform(t.sub) : GEMM_BM;
            decode_gemm_item(it, (m + sub - 1) / sub, syrk, rb, cb);
            const int r0 = rb * sub, c0 = cb * sub;
            // accumulate mode: one lock word per 128x128 sub-tile (16 per tile, shared beyond 4x4 sub-tiles)
            int32_t* lock = nullptr;
            if constexpr ((VM & V_ACC) != 0) {
                if (t.accum) lock = M.locks + ((long)(i + (long)j * nt) * 16 + (it & 15));
            } else if (t.accum) {
                return false;
            }
#define TTAD_GEMM_ITEM(TS_, PREC_)                                                                                 \
    if constexpr ((VM & V_ACC) != 0) {                                                                             \
        if (lock) {                                                                                                \
            gemm_acc_call<TS_, PREC_, VM>((const TS_*)opA, m, (const TS_*)opB, n, (TS_*)opC, m, m, n, K, r0, c0,  \
                                          syrk, lock, err, spin_limit, lds);                                       \
            return true;                                                                                           \
        }                                                                                                          \
    }                                                                                                              \
    if constexpr (GOPS) {                                                                                          \
        constexpr bool fold = sizeof(TS_) == 4 && PREC_ != P_BF16X3;                                               \
        if (sub == GEMM_BS)                                                                                        \
            gemm_small_call<TS_, PREC_, VM>((const TS_*)opA, (const TS_*)opB, (TS_*)opC, m, n, K, r0, c0, syrk,    \
                                            lds, opPA, opPB);                                                      \
        else if (fold && span > 1)                                                                                 \
            gemm_call<TS_, PREC_, VM, fold>(go, span, r0, c0, syrk, lds);                                          \
        else                                                                                                       \
            gemm_call<TS_, PREC_, VM, false>(go, span, r0, c0, syrk, lds);                                         \
    } else {                                                                                                       \
        item_gemm<TS_, PREC_>((const TS_*)opA, m, (const TS_*)opB, n, (TS_*)opC, m, m, n, K, r0, c0, syrk, -1.0,   \
                              1.0, lds, opPA, opPB);                                                               \
    }                                                                                                              \
    return true;
            // Products read C after the last K-chunk: measured faster than reading it with the first chunk
            // for FP64 (factorization at n = 32768: 246.7 -> 229.4 ms) and for bf16x3 items (11 %).
            if constexpr ((VM & V_F64S) != 0)
                if (t.prec == P_F64) { TTAD_GEMM_ITEM(double, P_F64) }
            if constexpr ((VM & V_G32) != 0)
                if (t.prec == P_F32) { TTAD_GEMM_ITEM(float, P_F32) }
            if constexpr ((VM & V_GBF16) != 0)
                if (t.prec == P_BF16) { TTAD_GEMM_ITEM(float, P_BF16) }
            if constexpr ((VM & V_GBF16X3) != 0)
                if (t.prec == P_BF16X3) { TTAD_GEMM_ITEM(float, P_BF16X3) }
#undef TTAD_GEMM_ITEM
            return false;
        }
        default:
            return false;
    }
}

}  // namespace ttad
