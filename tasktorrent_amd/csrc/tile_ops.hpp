// Device tile operations of the Cholesky DAG, written for gfx950 (CDNA4):
// one workgroup = 256 threads = 4 wave64; all products on MFMA 16x16 tiles.
//
// Replaces the CPU BLAS/LAPACK task bodies of miniapp/dense_cholesky/2d_cholesky.cpp:
//   LAPACKE_dpotrf('L')                       :319      -> item_potrf
//   cblas_dtrsm(Right, Lower, Trans, NonUnit)  :404-405  -> item_trsm
//   cblas_dsyrk(Lower, NoTrans, -1, ., beta)   :490-491  -> item_gemm(syrk=true)
//   cblas_dgemm(NoTrans, Trans, -1, ., beta)   :493-494  -> item_gemm
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <type_traits>
#include "ttad_types.hpp"

namespace ttad {

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef short s8_t __attribute__((ext_vector_type(8)));

// Device memory accesses of the item code go through address-space-1 pointers. Tile
// pointers reach it through tables in memory, so the compiler sees generic pointers and
// emits flat instructions, which count against the LDS wait counter as well: every LDS
// wait of a GEMM loop would then also wait for the prefetched loads of the next chunk.
#define TTAD_GLOBAL __attribute__((address_space(1)))
template <typename T> __device__ __forceinline__ const TTAD_GLOBAL T* gmem(const T* p) {
    return (const TTAD_GLOBAL T*)p;
}
template <typename T> __device__ __forceinline__ TTAD_GLOBAL T* gmem(T* p) { return (TTAD_GLOBAL T*)p; }
// A value the whole wave holds, moved to scalar registers: values loaded from task records in global
// memory are vector loads (the executors write global memory), so the compiler cannot tell they are
// uniform; address arithmetic on them would otherwise be 64-bit vector work per lane.
__device__ __forceinline__ int wave_uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
template <typename T> __device__ __forceinline__ T* wave_uniform(T* p) {
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return (T*)(((unsigned long long)hi << 32) | lo);
}

// Agent-scope release that has completed when it returns: buffer_wbl2 starts the write-back of this XCD's L2 and
// counts in vmcnt, but the compiler drops the wait that belongs behind it wherever it sees no other memory operation
// of this wave outstanding (after an explicit vmcnt(0), or after a barrier), and the store or atomic that announces
// the data would then pass the write-back. Every announcement therefore goes through this and is relaxed itself.
__device__ __forceinline__ void release_agent() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Every store of this wave has reached the L2 (vmcnt(0) expcnt(7) lgkmcnt(15); gfx9 counts stores in vmcnt). Where one
// thread releases what a whole workgroup has stored, every wave waits like this in front of the barrier behind which the
// thread does: the barrier itself waits for no store, and release_agent only for those of its own wave.
__device__ __forceinline__ void stores_done() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// The workgroup's dynamic LDS as a pointer in a scalar register. In a function called out of line its base is read
// from a table in memory, and the compiler reads it again at every use it cannot hoist (a memory round trip in front
// of LDS accesses on the critical path); the offset is opaque here, so it is read once.
__device__ __forceinline__ char* lds_uniform(char* p) {
    typedef __attribute__((address_space(3))) char lds_char;
    unsigned off = (unsigned)(unsigned long long)(lds_char*)p;
    asm volatile("" : "+v"(off));
    return (char*)(lds_char*)(unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane(off);
}

// ---------------------------------------------------------------------------
// MFMA 16x16 primitives. Operand layouts (lane l of the wave):
//   f64/f32 16x16x4 : A[m = l%16][k = l/16], B[k = l/16][n = l%16]
//   bf16   16x16x32 : A[m = l%16][k = 8(l/16)+e], B[k = 8(l/16)+e][n = l%16], e = 0..7
//   result f32/bf16 : D[m = 4(l/16)+r][n = l%16], r = 0..3
//   result f64      : D[m = (l/16)+4r][n = l%16], r = 0..3  (measured on gfx950)
// ---------------------------------------------------------------------------
template <typename TC> struct Mfma;
template <> struct Mfma<double> {
    typedef d4_t acc_t;
    static constexpr int KSTEP = 4;
    static __device__ __forceinline__ int row(int lane, int r) { return (lane >> 4) + 4 * r; }
    static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
};
template <> struct Mfma<float> {
    typedef f4_t acc_t;
    static constexpr int KSTEP = 4;
    static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
    static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
};

template <typename T> __device__ __forceinline__ T zero_val() { return T(0); }
constexpr int cmax(int a, int b) { return a > b ? a : b; }

// 16-byte register vectors of a storage type (aligned: LDS side; u: global side, element-aligned).
template <typename T> struct V16;
template <> struct V16<double> {
    static constexpr int N = 2;
    typedef double t __attribute__((ext_vector_type(2)));
    typedef double u __attribute__((ext_vector_type(2), aligned(8)));
};
template <> struct V16<float> {
    static constexpr int N = 4;
    typedef float t __attribute__((ext_vector_type(4)));
    typedef float u __attribute__((ext_vector_type(4), aligned(4)));
};

// What a product does after the last K-chunk of each pair of operands.
struct NoFold {
    static constexpr bool on = false;
    __device__ void operator()() const {}
};
template <typename F> struct FoldWith {
    static constexpr bool on = true;
    F f;
    __device__ __forceinline__ void operator()() const { f(); }
};

// ---------------------------------------------------------------------------
// acc (BM x BN) += A(BM x K) * B(BN x K)^T with A, B column-major (lda, ldb),
// rows >= mv of A and rows >= nv of B read as zero. TA/TB are storage types,
// TC the MFMA type; conversion happens on the register -> LDS path.
// 2x2 waves, each wave owns a (BM/2) x (BN/2) block of 16x16 MFMA tiles.
// K is staged through two LDS buffers in chunks of BK: while the MFMAs consume
// chunk c, chunk c+1 goes from registers to the other buffer and the global
// loads of chunk c+2 are in flight (one barrier per chunk).
// VEC: each lane loads 16 bytes (2 FP64 / 4 FP32 consecutive rows of a column) and
//      stores them to LDS in one instruction (TA = TB = TC).
// SWAP: the MFMA takes B's block as its first operand, so that a lane's results lie
//      along a column of the output (row = lane % 16): C is then read and written in
//      16-row segments instead of 16 scattered columns.
// ---------------------------------------------------------------------------
// WR: waves stacked along the rows (2: 2x2 waves; 4: each wave owns BM/4 full rows).
template <typename TA, typename TB, typename TC, int BM, int BN, int BK, bool VEC = false, bool SWAP = false, int WR = 2>
struct GemmNT {
    static constexpr int NVA = VEC ? V16<TA>::N : 1;  // rows per lane load
    static constexpr int NVB = VEC ? V16<TB>::N : 1;
    static constexpr int PA = BM + (NVA > 2 ? NVA : 2);  // LDS row pitch (16-byte multiple when VEC)
    static constexpr int PB = BN + (NVB > 2 ? NVB : 2);
    static constexpr int WC = 4 / WR;             // waves along the columns
    static constexpr int WM = BM / (16 * WR);     // 16x16 blocks per wave
    static constexpr int WN = BN / (16 * WC);
    static constexpr int LA = BM / NVA;          // lanes per column of the A chunk
    static constexpr int LB = BN / NVB;
    static constexpr int KS_A = NTHREADS / LA;   // columns per load round
    static constexpr int KS_B = NTHREADS / LB;
    static constexpr int EA = BK / KS_A;         // loads per thread per chunk
    static constexpr int EB = BK / KS_B;
    static constexpr int STAGE = BK * (PA + PB);  // TC elements of one LDS buffer
    static constexpr int LDS_BYTES = 2 * STAGE * (int)sizeof(TC);
    typedef typename Mfma<TC>::acc_t acc_t;
    typedef std::conditional_t<VEC, typename V16<TA>::t, TA> RA;
    typedef std::conditional_t<VEC, typename V16<TB>::t, TB> RB;
    static_assert(NTHREADS % LA == 0 && NTHREADS % LB == 0 && BK % KS_A == 0 && BK % KS_B == 0, "tile/thread mismatch");
    static_assert(!VEC || (std::is_same<TA, TC>::value && std::is_same<TB, TC>::value), "VEC stages without conversion");
    static_assert(BK % 4 == 0, "BK is a multiple of the MFMA k-step");

    static __device__ __forceinline__ void zero(acc_t (&acc)[WM][WN]) {
#pragma unroll
        for (int a = 0; a < WM; a++)
#pragma unroll
            for (int b = 0; b < WN; b++) acc[a][b] = acc_t{0, 0, 0, 0};
    }
    // Element (row, col) of the output block held by this lane in acc[a][b][r].
    static __device__ __forceinline__ int row_of(int a, int r) {
        const int lane = threadIdx.x & 63, wr = (threadIdx.x >> 6) / WC;
        return wr * (WM * 16) + a * 16 + (SWAP ? (lane & 15) : Mfma<TC>::row(lane, r));
    }
    static __device__ __forceinline__ int col_of(int b, int r) {
        const int lane = threadIdx.x & 63, wc = (threadIdx.x >> 6) % WC;
        return wc * (WN * 16) + b * 16 + (SWAP ? Mfma<TC>::row(lane, r) : (lane & 15));
    }

    // Thread tid stages rows NV*(tid % L) .. +NV-1 of every (NTHREADS/L)-th column of a chunk:
    // one wave instruction reads whole columns (coalesced).
    template <typename T, typename R, int E, int NV, int L, int KS>
    static __device__ __forceinline__ void load_chunk(R (&reg)[E], const T* __restrict__ base, long ld, int nvalid,
                                                      int k0, int K) {
        const int row = NV * ((int)threadIdx.x % L), kc = (int)threadIdx.x / L;
        if (nvalid >= L * NV && k0 + KS * E <= K) {  // whole chunk inside (uniform): no guards
#pragma unroll
            for (int s = 0; s < E; s++) {
                const TTAD_GLOBAL T* p = gmem(base) + row + (long)(k0 + kc + s * KS) * ld;
                if constexpr (NV == 1) reg[s] = *p;
                else reg[s] = *reinterpret_cast<const TTAD_GLOBAL typename V16<T>::u*>(p);
            }
            return;
        }
#pragma unroll
        for (int s = 0; s < E; s++) {
            const int kk = k0 + kc + s * KS;
            const TTAD_GLOBAL T* p = gmem(base) + row + (long)kk * ld;
            if constexpr (NV == 1) {
                reg[s] = (row < nvalid && kk < K) ? *p : T(0);
            } else {
#pragma unroll
                for (int q = 0; q < NV; q++) reg[s][q] = (kk < K && row + q < nvalid) ? p[q] : T(0);
            }
        }
    }
    template <typename R, int E, int NV, int L, int KS, int P>
    static __device__ __forceinline__ void store_chunk(TC* __restrict__ S, const R (&reg)[E]) {
        const int row = NV * ((int)threadIdx.x % L), kc = (int)threadIdx.x / L;
#pragma unroll
        for (int s = 0; s < E; s++) {
            TC* q = S + (kc + s * KS) * P + row;
            if constexpr (NV == 1) *q = (TC)reg[s];
            else *reinterpret_cast<R*>(q) = reg[s];
        }
    }
    static __device__ __forceinline__ void load(RA (&ra)[EA], RB (&rb)[EB], const TA* A, long lda, int mv, const TB* B,
                                                long ldb, int nv, int k0, int K) {
        load_chunk<TA, RA, EA, NVA, LA, KS_A>(ra, A, lda, mv, k0, K);
        load_chunk<TB, RB, EB, NVB, LB, KS_B>(rb, B, ldb, nv, k0, K);
    }
    static __device__ __forceinline__ void store(TC* __restrict__ S, const RA (&ra)[EA], const RB (&rb)[EB]) {
        store_chunk<RA, EA, NVA, LA, KS_A, PA>(S, ra);
        store_chunk<RB, EB, NVB, LB, KS_B, PB>(S + BK * PA, rb);
    }

    static __device__ __forceinline__ void run(acc_t (&acc)[WM][WN], const TA* __restrict__ A, long lda, int mv,
                                               const TB* __restrict__ B, long ldb, int nv, int K, char* lds) {
        run(acc, A, lda, mv, B, ldb, nv, K, lds, nullptr, 0, 0, 0, NoFold());
    }

    static __device__ __forceinline__ void compute(acc_t (&acc)[WM][WN], const TC* __restrict__ S, int lane, int wr,
                                                   int wc) {
        const TC* As = S + wr * (WM * 16) + (lane & 15);
        const TC* Bs = S + BK * PA + wc * (WN * 16) + (lane & 15);
#pragma unroll 4
        for (int ks = 0; ks < BK / 4; ks++) {
            const int kr = ks * 4 + (lane >> 4);
            TC av[WM], bv[WN];
#pragma unroll
            for (int a = 0; a < WM; a++) av[a] = As[kr * PA + a * 16];
#pragma unroll
            for (int b = 0; b < WN; b++) bv[b] = Bs[kr * PB + b * 16];
#pragma unroll
            for (int a = 0; a < WM; a++)
#pragma unroll
                for (int b = 0; b < WN; b++)
                    acc[a][b] = SWAP ? Mfma<TC>::mma(bv[b], av[a], acc[a][b]) : Mfma<TC>::mma(av[a], bv[b], acc[a][b]);
        }
    }

    // Starts and ends with a workgroup barrier: the caller may use `lds` before and after.
    // more > 0: further pairs of operands steps[0 .. more - 1] of K columns each (same shapes; their rows ra0 and rb0 on)
    // follow in the same pipeline; K is then a multiple of BK.
    // fold: called after the last chunk of each pair.
    template <typename Fold>
    static __device__ __forceinline__ void run(acc_t (&acc)[WM][WN], const TA* __restrict__ A, long lda, int mv,
                                               const TB* __restrict__ B, long ldb, int nv, int K, char* lds,
                                               const GemmOperands* __restrict__ steps, int more, int ra0, int rb0,
                                               Fold fold) {
        TC* S0 = reinterpret_cast<TC*>(lds);
        const int tid = threadIdx.x;
        const int lane = tid & 63, w = tid >> 6, wr = w / WC, wc = w % WC;
        const int K0 = K;
        int next = K0;  // the first column of the next pair, which is addressed as if it followed the first
        K += more * K0;
        auto advance = [&](int k0) {
            if (more > 0 && k0 == next && k0 < K) {
                A = static_cast<const TA*>(wave_uniform(steps->A)) + ra0 - (long)k0 * lda;
                B = static_cast<const TB*>(wave_uniform(steps->B)) + rb0 - (long)k0 * ldb;
                steps++;
                next += K0;
            }
        };
        const int nchunks = (K + BK - 1) / BK;
        __syncthreads();
        if (nchunks == 0) return;
        RA ra[EA];
        RB rb[EB];
        load(ra, rb, A, lda, mv, B, ldb, nv, 0, K);
        store(S0, ra, rb);
        advance(BK);
        if (nchunks > 1) load(ra, rb, A, lda, mv, B, ldb, nv, BK, K);
        __syncthreads();
        int done = K0;
        for (int c = 0; c < nchunks; c++) {
            compute(acc, S0 + (c & 1) * STAGE, lane, wr, wc);
            if constexpr (Fold::on)
                if ((c + 1) * BK == done) {
                    fold();
                    done += K0;
                }
            if (c + 1 < nchunks) {
                // the other buffer was last read in chunk c-1, before the previous barrier
                store(S0 + ((c + 1) & 1) * STAGE, ra, rb);
                if (c + 2 < nchunks) {
                    advance((c + 2) * BK);
                    load(ra, rb, A, lda, mv, B, ldb, nv, (c + 2) * BK, K);
                }
            }
            __syncthreads();
        }
    }
};

// ---------------------------------------------------------------------------
// BF16 inputs, FP32 accumulation: acc (BM x BN) += bf16(A) * bf16(B)^T.
// LDS holds bf16 in [row][k] order so that one lane reads its 8 consecutive k
// values with a single 16-byte load. Raw FP32 values are prefetched one chunk
// ahead in registers and converted (v_cvt_pk_bf16_f32, round to nearest even)
// on their way into the LDS buffer not being read; two buffers, one barrier per chunk.
// ---------------------------------------------------------------------------
// SPLIT = true: each FP32 operand x is split into hi = bf16(x) and lo = bf16(x - hi)
// and the product accumulates hi*hi + hi*lo + lo*hi (three MFMAs), which keeps about
// 16 significant bits of every operand (Henry, Tang, Heinecke, "Leveraging the
// bfloat16 artificial intelligence datatype for higher-precision computations", 2019).
typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
typedef float f2_t __attribute__((ext_vector_type(2)));
typedef unsigned u4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned pack_bf16x2(float a, float b) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector((f2_t){a, b}, bf2_t));
}

template <typename TA, int BM, int BN, bool SPLIT = false, bool SWAP = false>
struct GemmNTbf16 {
    // K-chunk: 64 (one plane), 32 with the hi/lo planes, so that both fit two workgroups per
    // CU (72 KB of LDS). Rows of 72 elements (144 B) are read 16 bytes at a time; rows of 36
    // (72 B, the split planes) 8 bytes at a time; both pitches spread 16 rows over distinct banks.
    static constexpr int BK = SPLIT ? 32 : 64;
    static constexpr int PK = SPLIT ? BK + 4 : BK + 8;  // bf16 elements per LDS row
    static constexpr bool NARROW = (PK * 2) % 16 != 0;  // LDS accesses in 8-byte halves
    static constexpr int WM = BM / 32;
    static constexpr int WN = BN / 32;
    static constexpr int NP = SPLIT ? 2 : 1;  // hi (and lo) planes
    static constexpr int STAGE = NP * (BM + BN) * PK;  // bf16 elements of one LDS buffer
    static constexpr int LDS_BYTES = 2 * STAGE * 2;
    typedef f4_t acc_t;
    // each thread owns groups of 8 consecutive k of one row
    static constexpr int GA = BM * (BK / 8) / NTHREADS;
    static constexpr int GB = BN * (BK / 8) / NTHREADS;
    static_assert(GA * NTHREADS == BM * (BK / 8) && GB * NTHREADS == BN * (BK / 8), "tile/thread mismatch");

    static __device__ __forceinline__ void run(acc_t (&acc)[WM][WN], const TA* __restrict__ A, long lda, int mv,
                                               const TA* __restrict__ B, long ldb, int nv, int K, char* lds) {
        run(acc, A, lda, mv, B, ldb, nv, K, lds, nullptr, 0, 0, 0, NoFold());
    }
    static __device__ __forceinline__ void zero(acc_t (&acc)[WM][WN]) {
#pragma unroll
        for (int a = 0; a < WM; a++)
#pragma unroll
            for (int b = 0; b < WN; b++) acc[a][b] = acc_t{0, 0, 0, 0};
    }
    static __device__ __forceinline__ int row_of(int a, int r) {
        const int lane = threadIdx.x & 63, wr = (threadIdx.x >> 6) >> 1;
        return wr * (WM * 16) + a * 16 + (SWAP ? (lane & 15) : 4 * (lane >> 4) + r);
    }
    static __device__ __forceinline__ int col_of(int b, int r) {
        const int lane = threadIdx.x & 63, wc = (threadIdx.x >> 6) & 1;
        return wc * (WN * 16) + b * 16 + (SWAP ? 4 * (lane >> 4) + r : (lane & 15));
    }
    static __device__ __forceinline__ f4_t mma(s8_t a, s8_t b, f4_t c) {
        return SWAP ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, c, 0, 0, 0)
                    : __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }

    // full: the whole chunk is inside the operand (uniform), so the loads need no guards; the
    // guarded form, one exec-masked branch per load, is kept for edge chunks. base is the
    // operand's (uniform) first row and kfirst is uniform over the wave, so each column's address
    // is a scalar base plus this lane's 32-bit row offset: no per-lane 64-bit address is kept per
    // column (those spilled, and a reload from scratch waits for every load in flight, which made
    // the one-chunk prefetch synchronous).
    template <int G, int GS>
    static __device__ __forceinline__ void load_raw(float (&r)[G][8], const TA* __restrict__ base, long ld, int row,
                                                    bool row_ok, int kfirst, int K, bool full) {
        const TTAD_GLOBAL TA* gb = gmem(base);
        if (full) {
#pragma unroll
            for (int s = 0; s < G; s++) {
                const int k = kfirst + s * GS * 8;
#pragma unroll
                for (int q = 0; q < 8; q++) r[s][q] = (float)(gb + (long)(k + q) * ld)[row];
            }
            return;
        }
#pragma unroll
        for (int s = 0; s < G; s++) {
            const int k = kfirst + s * GS * 8;
#pragma unroll
            for (int q = 0; q < 8; q++)
                r[s][q] = (row_ok && k + q < K) ? (float)(gb + (long)(k + q) * ld)[row] : 0.0f;
        }
    }

    template <int G, int GS>
    static __device__ __forceinline__ void store_planes(unsigned short* __restrict__ hi_plane,
                                                        unsigned short* __restrict__ lo_plane, const float (&r)[G][8],
                                                        int row, int g0) {
#pragma unroll
        for (int s = 0; s < G; s++) {
            u4_t h, l;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float x0 = r[s][2 * q], x1 = r[s][2 * q + 1];
                const unsigned hp = pack_bf16x2(x0, x1);
                h[q] = hp;
                if constexpr (SPLIT)
                    l[q] = pack_bf16x2(x0 - __uint_as_float(hp << 16), x1 - __uint_as_float(hp & 0xffff0000u));
            }
            const int off = row * PK + (g0 + s * GS) * 8;
            if constexpr (NARROW) {
                typedef unsigned u2_t __attribute__((ext_vector_type(2)));
                *reinterpret_cast<u2_t*>(hi_plane + off) = u2_t{h[0], h[1]};
                *reinterpret_cast<u2_t*>(hi_plane + off + 4) = u2_t{h[2], h[3]};
                if constexpr (SPLIT) {
                    *reinterpret_cast<u2_t*>(lo_plane + off) = u2_t{l[0], l[1]};
                    *reinterpret_cast<u2_t*>(lo_plane + off + 4) = u2_t{l[2], l[3]};
                }
            } else {
                *reinterpret_cast<u4_t*>(hi_plane + off) = h;
                if constexpr (SPLIT) *reinterpret_cast<u4_t*>(lo_plane + off) = l;
            }
        }
    }

    // 8 consecutive bf16 (one lane's k-group, already split) into LDS
    static __device__ __forceinline__ void put8(unsigned short* p, u4_t v) {
        if constexpr (NARROW) {
            typedef unsigned u2_t __attribute__((ext_vector_type(2)));
            *reinterpret_cast<u2_t*>(p) = u2_t{v[0], v[1]};
            *reinterpret_cast<u2_t*>(p + 4) = u2_t{v[2], v[3]};
        } else {
            *reinterpret_cast<u4_t*>(p) = v;
        }
    }

    // 8 consecutive bf16 (one lane's k-group) from LDS
    static __device__ __forceinline__ s8_t ld8(const unsigned short* p) {
        if constexpr (NARROW) {
            typedef short s4_t __attribute__((ext_vector_type(4)));
            const s4_t a = *reinterpret_cast<const s4_t*>(p), b = *reinterpret_cast<const s4_t*>(p + 4);
            return s8_t{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
        } else {
            return *reinterpret_cast<const s8_t*>(p);
        }
    }
    static __device__ __forceinline__ void compute(acc_t (&acc)[WM][WN], const unsigned short* __restrict__ S,
                                                   int lane, int wr, int wc) {
        const unsigned short* As = S;
        const unsigned short* Bs = As + BM * PK;
        const unsigned short* Al = Bs + BN * PK;
        const unsigned short* Bl = Al + BM * PK;
#pragma unroll 1  // one k-step's hi/lo operands live at a time (register budget of the executors)
        for (int ks = 0; ks < BK / 32; ks++) {
            const int kg = ks * 32 + (lane >> 4) * 8;
            s8_t av[WM], bv[WN];
#pragma unroll
            for (int a = 0; a < WM; a++)
                av[a] = ld8(As + (wr * (WM * 16) + a * 16 + (lane & 15)) * PK + kg);
#pragma unroll
            for (int b = 0; b < WN; b++)
                bv[b] = ld8(Bs + (wc * (WN * 16) + b * 16 + (lane & 15)) * PK + kg);
#pragma unroll
            for (int a = 0; a < WM; a++)
#pragma unroll
                for (int b = 0; b < WN; b++)
                    acc[a][b] = mma(av[a], bv[b], acc[a][b]);
            if constexpr (SPLIT) {
                s8_t avl[WM], bvl[WN];
#pragma unroll
                for (int a = 0; a < WM; a++)
                    avl[a] = ld8(Al + (wr * (WM * 16) + a * 16 + (lane & 15)) * PK + kg);
#pragma unroll
                for (int b = 0; b < WN; b++)
                    bvl[b] = ld8(Bl + (wc * (WN * 16) + b * 16 + (lane & 15)) * PK + kg);
#pragma unroll
                for (int a = 0; a < WM; a++)
#pragma unroll
                    for (int b = 0; b < WN; b++) {
                        acc[a][b] = mma(av[a], bvl[b], acc[a][b]);
                        acc[a][b] = mma(avl[a], bv[b], acc[a][b]);
                    }
            }
        }
    }

    // Starts and ends with a workgroup barrier: the caller may use `lds` before and after.
    // steps, more, ra0, rb0, fold as GemmNT::run.
    template <typename Fold>
    static __device__ __forceinline__ void run(acc_t (&acc)[WM][WN], const TA* __restrict__ A, long lda, int mv,
                               const TA* __restrict__ B, long ldb, int nv, int K, char* lds,
                               const GemmOperands* __restrict__ steps, int more, int ra0, int rb0, Fold fold) {
        const int K0 = K;
        int next = K0;
        K += more * K0;
        auto advance = [&](int k0) {
            if (more > 0 && k0 == next && k0 < K) {
                A = static_cast<const TA*>(wave_uniform(steps->A)) + ra0 - (long)k0 * lda;
                B = static_cast<const TA*>(wave_uniform(steps->B)) + rb0 - (long)k0 * ldb;
                steps++;
                next += K0;
            }
        };
        unsigned short* S0 = reinterpret_cast<unsigned short*>(lds);
        const int tid = threadIdx.x;
        const int lane = tid & 63, w = tid >> 6, wr = w >> 1, wc = w & 1;
        // thread -> fixed row (tid % BM) and k-groups of 8 (tid / BM + s * NTHREADS / BM); BM and BN are
        // multiples of the wave size, so a_g and b_g are the same over a wave
        static_assert(BM % 64 == 0 && BN % 64 == 0, "k-group of a thread must be uniform over its wave");
        const int a_row = tid % BM, b_row = tid % BN;
        const int a_g = __builtin_amdgcn_readfirstlane(tid / BM), b_g = __builtin_amdgcn_readfirstlane(tid / BN);
        const bool a_ok = a_row < mv, b_ok = b_row < nv;
        const int nchunks = (K + BK - 1) / BK;
        __syncthreads();
        if (nchunks == 0) return;
        float ra[GA][8], rb[GB][8];
        auto stage = [&](unsigned short* S) {
            store_planes<GA, NTHREADS / BM>(S, S + (BM + BN) * PK, ra, a_row, a_g);
            store_planes<GB, NTHREADS / BN>(S + BM * PK, S + (BM + BN) * PK + BM * PK, rb, b_row, b_g);
        };
        // a chunk is full when both operands have all their rows and the chunk lies inside K
        const bool rows_full = __builtin_amdgcn_readfirstlane((int)(mv >= BM && nv >= BN)) != 0;
        auto full = [&](int k0) { return rows_full && k0 + BK <= K; };
        load_raw<GA, NTHREADS / BM>(ra, A, lda, a_row, a_ok, a_g * 8, K, full(0));
        load_raw<GB, NTHREADS / BN>(rb, B, ldb, b_row, b_ok, b_g * 8, K, full(0));
        stage(S0);
        if (nchunks > 1) {
            advance(BK);
            load_raw<GA, NTHREADS / BM>(ra, A, lda, a_row, a_ok, BK + a_g * 8, K, full(BK));
            load_raw<GB, NTHREADS / BN>(rb, B, ldb, b_row, b_ok, BK + b_g * 8, K, full(BK));
        }
        __syncthreads();
        int done = K0;
        for (int c = 0; c < nchunks; c++) {
            compute(acc, S0 + (c & 1) * STAGE, lane, wr, wc);
            if constexpr (Fold::on)
                if ((c + 1) * BK == done) {
                    fold();
                    done += K0;
                }
            if (c + 1 < nchunks) {
                stage(S0 + ((c + 1) & 1) * STAGE);
                if (c + 2 < nchunks) {
                    const int k0 = (c + 2) * BK;
                    advance(k0);
                    load_raw<GA, NTHREADS / BM>(ra, A, lda, a_row, a_ok, k0 + a_g * 8, K, full(k0));
                    load_raw<GB, NTHREADS / BN>(rb, B, ldb, b_row, b_ok, k0 + b_g * 8, K, full(k0));
                }
            }
            __syncthreads();
        }
    }

    // As run() for SPLIT with BM x BN fully inside both operands and K % BK == 0, from operands
    // already split into bf16 planes (plane_granule layout; PA and PB point at the granule of the
    // item's first row, arows / brows are the tiles' row counts). Each thread moves whole 16-byte
    // granules, so a chunk costs 4 loads per operand and no conversion; the LDS buffers receive
    // exactly what run() would store from the FP32 values the planes were split from.
    // more > 0: the planes of steps[0 .. more - 1] follow (their rows ra0 and rb0 on).
    template <typename Fold>
    static __device__ __forceinline__ void run_planes(acc_t (&acc)[WM][WN], const u4_t* __restrict__ PA, int arows,
                                                      const u4_t* __restrict__ PB, int brows, int K, char* lds,
                                                      const GemmOperands* __restrict__ steps, int more, int ra0,
                                                      int rb0, Fold fold) {
        static_assert(SPLIT && BK == 32, "plane chunks are 32 columns of hi and lo");
        unsigned short* S0 = reinterpret_cast<unsigned short*>(lds);
        const int tid = threadIdx.x;
        const int lane = tid & 63, w = tid >> 6, wr = w >> 1, wc = w & 1;
        const int a_row = tid % BM, b_row = tid % BN;
        const int a_g = __builtin_amdgcn_readfirstlane(tid / BM), b_g = __builtin_amdgcn_readfirstlane(tid / BN);
        const int nc0 = wave_uniform(K / BK), nchunks = wave_uniform(nc0 * (1 + more));
        int next = nc0;
        arows = wave_uniform(arows);
        brows = wave_uniform(brows);
        __syncthreads();
        if (nchunks == 0) return;
        u4_t ra[GA][2], rb[GB][2];
        // uniform bases of the next chunk's granules, moved on with each fetch, plus this lane's 32-bit row offset
        const TTAD_GLOBAL u4_t* ga = gmem(wave_uniform(PA));
        const TTAD_GLOBAL u4_t* gb = gmem(wave_uniform(PB));
        auto fetch = [&](int c) {
            if (more > 0 && c == next) {
                ga = gmem(static_cast<const u4_t*>(wave_uniform(steps->PA)) + ra0);
                gb = gmem(static_cast<const u4_t*>(wave_uniform(steps->PB)) + rb0);
                steps++;
                next += nc0;
            }
#pragma unroll
            for (int s = 0; s < GA; s++)
#pragma unroll
                for (int p = 0; p < 2; p++)
                    ra[s][p] = (ga + plane_granule(0, p, a_g + s * (NTHREADS / BM), 0, arows))[a_row];
#pragma unroll
            for (int s = 0; s < GB; s++)
#pragma unroll
                for (int p = 0; p < 2; p++)
                    rb[s][p] = (gb + plane_granule(0, p, b_g + s * (NTHREADS / BN), 0, brows))[b_row];
            ga += plane_granule(1, 0, 0, 0, arows);
            gb += plane_granule(1, 0, 0, 0, brows);
        };
        auto stage = [&](unsigned short* S) {
            unsigned short* Ah = S;
            unsigned short* Bh = S + BM * PK;
            unsigned short* Al = S + (BM + BN) * PK;
            unsigned short* Bl = Al + BM * PK;
#pragma unroll
            for (int s = 0; s < GA; s++) {
                const int off = a_row * PK + (a_g + s * (NTHREADS / BM)) * 8;
                put8(Ah + off, ra[s][0]);
                put8(Al + off, ra[s][1]);
            }
#pragma unroll
            for (int s = 0; s < GB; s++) {
                const int off = b_row * PK + (b_g + s * (NTHREADS / BN)) * 8;
                put8(Bh + off, rb[s][0]);
                put8(Bl + off, rb[s][1]);
            }
        };
        fetch(0);
        stage(S0);
        if (nchunks > 1) fetch(1);
        __syncthreads();
        int done = nc0;
        for (int c = 0; c < nchunks; c++) {
            compute(acc, S0 + (c & 1) * STAGE, lane, wr, wc);
            if constexpr (Fold::on)
                if (c + 1 == done) {
                    fold();
                    done += nc0;
                }
            if (c + 1 < nchunks) {
                stage(S0 + ((c + 1) & 1) * STAGE);
                if (c + 2 < nchunks) fetch(c + 2);
            }
            __syncthreads();
        }
    }
};

// Splits 4 consecutive FP32 values of a row (columns k .. k+3, k % 4 == 0) into the bf16 hi/lo planes
// of a tile of m rows (plane_granule layout), with the rounding GemmNTbf16 applies on its way to LDS.
__device__ __forceinline__ void store_split4(unsigned short* __restrict__ planes, int m, int row, int k, f4_t x) {
    typedef unsigned u2_t __attribute__((ext_vector_type(2)));
    const unsigned h01 = pack_bf16x2(x[0], x[1]), h23 = pack_bf16x2(x[2], x[3]);
    const unsigned l01 = pack_bf16x2(x[0] - __uint_as_float(h01 << 16), x[1] - __uint_as_float(h01 & 0xffff0000u));
    const unsigned l23 = pack_bf16x2(x[2] - __uint_as_float(h23 << 16), x[3] - __uint_as_float(h23 & 0xffff0000u));
    TTAD_GLOBAL unsigned short* g = gmem(planes);
    const long hi = plane_granule(k / 32, 0, (k % 32) / 8, row, m) * 8 + (k % 8);
    const long lo = plane_granule(k / 32, 1, (k % 32) / 8, row, m) * 8 + (k % 8);
    *reinterpret_cast<TTAD_GLOBAL u2_t*>(g + hi) = u2_t{h01, h23};
    *reinterpret_cast<TTAD_GLOBAL u2_t*>(g + lo) = u2_t{l01, l23};
}

// K-chunk of the 128x128 FP64/FP32 GEMM items: 16 FP64 / 32 FP32 columns, 65 KB of LDS for the
// two buffers, so that two workgroups share a CU: one's barriers, loads and C traffic overlap
// the other's MFMAs (FP64, m = n = 16384, K = 512: 43.5 TF/s with one 130 KB workgroup per CU,
// 53 TF/s with two; 66 TF/s with the 16-byte loads, coalesced C and C read up front).
// 64x64 items take chunks twice as long: they are used where latency counts (few items in flight), and each chunk costs
// a memory round trip.
template <typename TC, int BM = GEMM_BM> constexpr int gemm_bk() { return (sizeof(TC) == 8 ? 16 : 32) * (GEMM_BM / BM); }
// K-chunk of a TRSM item's update from the solved columns: each chunk waits for its loads (issued one chunk
// ahead), so fewer chunks cost fewer round trips. 64 FP32 columns fit the LDS of the FP32 executors; the FP64
// ones allow 32.
template <typename TS> constexpr int trsm_bk() { return sizeof(TS) == 4 ? 64 : 32; }

// ---------------------------------------------------------------------------
// GEMM / SYRK work item: C[r0:r0+128, c0:c0+128] = beta*C + alpha * A[r0:,:] B[c0:,:]^T
// over the valid part of an m x n tile, K = inner size. With syrk, only the
// lower triangle (global row >= global col) is written (dsyrk 'L').
// beta == 0 overwrites C without reading it (accumulate-mode temporaries).
// ---------------------------------------------------------------------------
// BM: rows and columns of the item, GEMM_BM or GEMM_BS.
// PA / PB (bf16x3 only; null = none): the bf16 split planes of the operand tiles (A and B with lda and ldb
// rows, plane_granule layout), used by items that lie wholly inside both with K % 32 == 0.
// steps, more: the operands of further steps of K columns each; C is then read and written once for all of them. K is a
// multiple of 64 then, and either all steps have planes or none. FOLD: C (beta = 1, alpha = -1) is read before the first
// step and each step's product is subtracted from it in registers, as items of one step would; without, the steps'
// products are summed first.
template <typename TS, int PREC, int BM = GEMM_BM, bool FOLD = false>
__device__ __forceinline__ void item_gemm(const TS* __restrict__ A, long lda, const TS* __restrict__ B, long ldb, TS* __restrict__ C,
                          long ldc, int m, int n, int K, int r0, int c0, bool syrk, double alpha, double beta,
                          char* lds, const void* PA = nullptr, const void* PB = nullptr,
                          const GemmOperands* __restrict__ steps = nullptr, int more = 0) {
    const int mv = min(BM, m - r0), nv = min(BM, n - c0);
    if (mv <= 0 || nv <= 0) return;
    auto body = [&](auto* gsel) {
        using G = typename std::remove_pointer<decltype(gsel)>::type;
        typedef typename G::acc_t acc_t;
        acc_t acc[G::WM][G::WN];
        auto owned = [&](int rr, int cc) { return rr < mv && cc < nv && (!syrk || r0 + rr >= c0 + cc); };
        const bool full = __builtin_amdgcn_readfirstlane(
                              (int)(mv == BM && nv == BM && (!syrk || r0 >= c0 + BM))) != 0;
        G::zero(acc);
        auto product = [&](auto fold) {
            if constexpr (PREC == P_BF16X3)
                if (PA && PB && mv == BM && nv == BM && K % G::BK == 0) {
                    G::run_planes(acc, static_cast<const u4_t*>(PA) + r0, (int)lda, static_cast<const u4_t*>(PB) + c0,
                                  (int)ldb, K, lds, steps, more, r0, c0, fold);
                    return;
                }
            G::run(acc, A + r0, lda, mv, B + c0, ldb, nv, K, lds, steps, more, r0, c0, fold);
        };
        if constexpr (FOLD) {
            acc_t tot[G::WM][G::WN];
#pragma unroll
            for (int a = 0; a < G::WM; a++)
#pragma unroll
                for (int b = 0; b < G::WN; b++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int rr = G::row_of(a, r), cc = G::col_of(b, r);
                        tot[a][b][r] = gmem(C)[(full || owned(rr, cc)) ? (r0 + rr) + (long)(c0 + cc) * ldc : 0];
                    }
            auto sub = [&]() {
#pragma unroll
                for (int a = 0; a < G::WM; a++)
#pragma unroll
                    for (int b = 0; b < G::WN; b++) {
                        tot[a][b] -= acc[a][b];
                        acc[a][b] = acc_t{0, 0, 0, 0};
                    }
            };
            product(FoldWith<decltype(sub)>{sub});
#pragma unroll
            for (int a = 0; a < G::WM; a++)
#pragma unroll
                for (int b = 0; b < G::WN; b++) acc[a][b] = tot[a][b];
            alpha = 1.0;
            beta = 0.0;
        } else {
            product(NoFold());
        }
        // C is read after the last K-chunk. Every load of a group of fragment rows is issued before any
        // store of the group: as far as the compiler knows a store may alias a later load, so a load and
        // a store per element in turn would cost one memory round trip per element (64 per item). Groups:
        // all of the item for FP32 tiles, one fragment row for FP64 (registers). Loads come from clamped addresses
        // (C[0] for elements not owned), so none waits under a branch; interior items (all of the
        // 128 x 128 owned) store without a condition.
        if constexpr (sizeof(TS) == 4) {
            // Interior FP32 items go through LDS (free after the K loop): a lane's results lie along a row,
            // C is column-major, so the accumulators are transposed in LDS and every thread then reads,
            // updates and writes 16 contiguous bytes of C per access (16 loads and 16 stores per thread
            // instead of 64 each). C is read first, so its latency overlaps the transposition.
            if (full) {
                constexpr int P = BM + 4;  // LDS column pitch: the 4 column groups of a wave hit distinct banks
                static_assert(BM * P * 4 <= G::LDS_BYTES, "transposed item fits the item's LDS");
                typedef typename V16<TS>::u f4u;
                TS* T = reinterpret_cast<TS*>(lds);
                constexpr int RL = BM / 4, CL = NTHREADS / RL;  // lanes along a column, columns per pass
                const int rg = threadIdx.x % RL, cl = threadIdx.x / RL;  // rows 4rg .. 4rg+3 of columns cl + CL j
                const long ldu = wave_uniform((int)ldc);
                TTAD_GLOBAL TS* base = gmem(C) + (r0 + 4 * rg) + (long)(c0 + cl) * ldu;
                constexpr int NJ = BM / CL;
                f4_t cv[NJ];
                if (beta != 0.0) {
#pragma unroll
                    for (int j = 0; j < NJ; j++) cv[j] = *reinterpret_cast<TTAD_GLOBAL f4u*>(base + CL * j * ldu);
                }
#pragma unroll
                for (int a = 0; a < G::WM; a++)
#pragma unroll
                    for (int b = 0; b < G::WN; b++)
#pragma unroll
                        for (int r = 0; r < 4; r++) T[G::col_of(b, r) * P + G::row_of(a, r)] = acc[a][b][r];
                __syncthreads();
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    const f4_t v = *reinterpret_cast<const f4_t*>(T + (cl + CL * j) * P + 4 * rg);
                    f4_t o;
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const double x = alpha * (double)v[r];
                        o[r] = (TS)(beta == 0.0 ? x : beta * (double)cv[j][r] + x);
                    }
                    *reinterpret_cast<TTAD_GLOBAL f4u*>(base + CL * j * ldu) = o;
                }
                __syncthreads();  // the caller may use lds again
                return;
            }
        }
        constexpr int AG = sizeof(TS) == 8 && BM == GEMM_BM ? 1 : G::WM;
#pragma unroll
        for (int a0 = 0; a0 < G::WM; a0 += AG) {
            TS cv[AG][G::WN][4];
            if (beta != 0.0) {
#pragma unroll
                for (int a = 0; a < AG; a++)
#pragma unroll
                    for (int b = 0; b < G::WN; b++)
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const int rr = G::row_of(a0 + a, r), cc = G::col_of(b, r);
                            const long off = (r0 + rr) + (long)(c0 + cc) * ldc;
                            cv[a][b][r] = gmem(C)[(full || owned(rr, cc)) ? off : 0];
                        }
            }
#pragma unroll
            for (int a = 0; a < AG; a++)
#pragma unroll
                for (int b = 0; b < G::WN; b++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int rr = G::row_of(a0 + a, r), cc = G::col_of(b, r);
                        const double v = alpha * (double)acc[a0 + a][b][r];
                        const TS o = (TS)(beta == 0.0 ? v : beta * (double)cv[a][b][r] + v);
                        if (full || owned(rr, cc)) gmem(C)[(r0 + rr) + (long)(c0 + cc) * ldc] = o;
                    }
        }
    };
    if constexpr (PREC == P_BF16 || PREC == P_BF16X3) {
        body((GemmNTbf16<TS, BM, BM, PREC == P_BF16X3, true>*)nullptr);
    } else {  // F64 tiles on FP64 MFMA, F32 tiles on FP32 MFMA
        body((GemmNT<TS, TS, TS, BM, BM, gemm_bk<TS, BM>(), true, true>*)nullptr);
    }
}

// Accumulate-mode GEMM / SYRK item (2d_cholesky.cpp:479-501 with beta = 0, then the ACCU task
// `*blocks[i+j*nb] += *Atmp`, :570, fused): the product is formed from zero and added into C while
// holding `lock`, the sub-tile's lock word (agent-scope acquire / release), so contributions of
// different k land in any order but one at a time. A lock wait gives up after spin_limit ticks or
// once *err is nonzero (and sets *err = 1 when it times out).
template <typename TS, int PREC>
__device__ __forceinline__ void item_gemm_acc(const TS* __restrict__ A, long lda, const TS* __restrict__ B, long ldb,
                                              TS* __restrict__ C, long ldc, int m, int n, int K, int r0, int c0,
                                              bool syrk, double alpha, int32_t* lock, int32_t* err,
                                              int64_t spin_limit, char* lds) {
    const int mv = min(GEMM_BM, m - r0), nv = min(GEMM_BM, n - c0);
    if (mv <= 0 || nv <= 0) return;
    auto body = [&](auto* gsel) {
        using G = typename std::remove_pointer<decltype(gsel)>::type;
        typedef typename G::acc_t acc_t;
        acc_t acc[G::WM][G::WN];
        G::zero(acc);
        G::run(acc, A + r0, lda, mv, B + c0, ldb, nv, K, lds);
        if (threadIdx.x == 0) {
            const int64_t t0 = (int64_t)wall_clock64();
            int expected = 0;
            while (!__hip_atomic_compare_exchange_strong(lock, &expected, 1, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_AGENT)) {
                expected = 0;
                if ((int64_t)wall_clock64() - t0 > spin_limit ||
                    __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) {
                    __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    break;
                }
                __builtin_amdgcn_s_sleep(2);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // the previous holder's additions
        }
        __syncthreads();
#pragma unroll
        for (int a = 0; a < G::WM; a++)
#pragma unroll
            for (int b = 0; b < G::WN; b++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int rr = G::row_of(a, r), cc = G::col_of(b, r);
                    if (rr < mv && cc < nv && (!syrk || r0 + rr >= c0 + cc)) {
                        TTAD_GLOBAL TS* p = gmem(C) + (r0 + rr) + (long)(c0 + cc) * ldc;
                        *p = (TS)((double)(*p) + alpha * (double)acc[a][b][r]);
                    }
                }
        stores_done();
        __syncthreads();
        if (threadIdx.x == 0) {
            release_agent();
            __hip_atomic_store(lock, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    };
    if constexpr (PREC == P_BF16 || PREC == P_BF16X3) {
        body((GemmNTbf16<TS, GEMM_BM, GEMM_BM, PREC == P_BF16X3, true>*)nullptr);
    } else {
        body((GemmNT<TS, TS, TS, GEMM_BM, GEMM_BM, gemm_bk<TS>(), true, true>*)nullptr);
    }
}

// Decode the (row block, col block) of GEMM/SYRK item `it` in a tile of tr x tc sub-tiles.
__device__ __forceinline__ void decode_gemm_item(int it, int tr, bool syrk, int& rb, int& cb) {
    if (!syrk) {
        rb = it % tr;
        cb = it / tr;
        return;
    }
    // lower-triangular enumeration, column-major: (c, r) with r >= c
    int c = 0, rem = it;
    while (rem >= tr - c) { rem -= tr - c; c++; }
    cb = c;
    rb = c + rem;
}

// ---------------------------------------------------------------------------
// 64x64 diagonal block in LDS (column-major, ld DP), blocked by 16: factor
// (lower Cholesky) and inverse. FP64 throughout. Padding rows/cols beyond `w`
// hold identity. 16-column panels are factored by one wave in registers;
// everything else is 16x16x16 products on FP64 MFMA, one block per wave.
// ---------------------------------------------------------------------------
constexpr int DP = DB + 1;

// acc += P Q (q_trans = false) or P Q^T (q_trans = true); P, Q 16x16 blocks in LDS, ld DP.
__device__ __forceinline__ d4_t mma16(d4_t acc, const double* P, const double* Q, bool q_trans) {
    const int lane = threadIdx.x & 63, m = lane & 15, kq = lane >> 4;
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int k = 4 * s + kq;
        const double b = q_trans ? Q[m + k * DP] : Q[k + m * DP];
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(P[m + k * DP], b, acc, 0, 0, 0);
    }
    return acc;
}
// R = sign * acc (acc in the FP64 MFMA result layout), or R += sign * acc.
__device__ __forceinline__ void put16(double* R, d4_t acc, double sign, bool add) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        double* p = R + ((lane >> 4) + 4 * r) + (lane & 15) * DP;
        *p = add ? *p + sign * acc[r] : sign * acc[r];
    }
}
// out = P T with T held in MFMA result registers (its row 4s + lane/16 is acc[s]: the B operand layout).
__device__ __forceinline__ d4_t mma16_reg(const double* P, d4_t T) {
    const int lane = threadIdx.x & 63, m = lane & 15, kq = lane >> 4;
    d4_t out = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; s++) out = __builtin_amdgcn_mfma_f64_16x16x4f64(P[m + (4 * s + kq) * DP], T[s], out, 0, 0, 0);
    return out;
}

// 1/x to about one ulp without the FP64 division sequence: the hardware reciprocal estimate refined by two
// Newton-Raphson steps r <- r + r (1 - x r), each of which doubles the number of correct bits. The POTRF
// diagonal blocks divide by every pivot in turn, so the division's latency is on the factorization's
// critical path.
__device__ __forceinline__ double rcp_nr(double x) {
    double r = __builtin_amdgcn_rcp(x);
    double e = __builtin_fma(-x, r, 1.0);
    r = __builtin_fma(r, e, r);
    e = __builtin_fma(-x, r, 1.0);
    return __builtin_fma(r, e, r);
}

// The value of lane SRC of each row of 16 lanes, in all 16 of them (one DPP move). Every lane has to be active.
template <int SRC>
__device__ __forceinline__ double row_value(double x) {
    const long v = __builtin_bit_cast(long, x);
    const long r = __builtin_amdgcn_update_dpp(v, v, 0x150 + SRC, 0xf, 0xf, true);  // row_newbcast
    return __builtin_bit_cast(double, r);
}
// f(K) for K = 0 .. N - 1 as a compile-time constant (DPP controls are immediates).
template <int K, int N, typename F>
__device__ __forceinline__ void for_const(const F& f) {
    if constexpr (K < N) {
        f(std::integral_constant<int, K>{});
        for_const<K + 1, N>(f);
    }
}

// Keeps the computation of x in front of this point.
__device__ __forceinline__ void hold(double& x) { asm volatile("" : "+v"(x)); }

// One wave factors a 16-column panel, a row per lane in a[]; p[] is the 16x16 diagonal block, row i in every lane with
// lane % 16 == i, so that pivot rows reach all lanes by moves within 16 lanes: a column costs no LDS round trip and no
// barrier. Lanes 0..15 hold the block's own rows in a[], every other lane a row b that becomes b L^{-T} (rows below
// the block; rows of the identity, which become L^{-T} itself). Unscaled elimination by the pivots' reciprocals, then
// the columns are scaled. Returns, in lane k < 16, whether pivot k is not positive.
__device__ __forceinline__ bool panel16(double (&p)[16], double (&a)[16]) {
    const int lane = threadIdx.x & 63, i = lane & 15;
    double dk = 1.0;  // lanes with i = k: pivot k
    double r = rcp_nr(row_value<0>(p[0]));
    for_const<0, 16>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        if (i == k) dk = p[k];
        const double lp = p[k] * r, la = a[k] * r;
        for_const<k + 1, 16>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            const double s = row_value<j>(p[k]);
            p[j] = __builtin_fma(-lp, s, p[j]);
            a[j] = __builtin_fma(-la, s, a[j]);
            // the next pivot's reciprocal, the chain of this loop, as soon as the pivot is final
            if constexpr (j == k + 1) r = rcp_nr(row_value<j>(p[j]));
        });
        // every update happens in its own column: put off to a later one, its operands would spill
#pragma unroll
        for (int j = k + 1; j < 16; j++) hold(a[j]);
        __builtin_amdgcn_sched_barrier(0);
    });
    const double s = sqrt(dk), rs = rcp_nr(s);
    for_const<0, 16>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        const double c = row_value<k>(rs);  // outside the selection: every lane takes part in the move
        a[k] = lane == k ? s : a[k] * c;
    });
    return !(dk > 0.0);
}

// X_KK = L_KK^{-1} for the 16x16 lower-triangular diagonal block at Lk (X block at Xk, all of it written), by one
// wave: lane r solves row r of the identity, e_r L^{-T}, which is column r of the inverse.
__device__ __forceinline__ void tri_inv16(const double* Lk, double* Xk) {
    const int lane = threadIdx.x & 63, i = lane & 15;
    double l[16], b[16];  // l: row i of the block
#pragma unroll
    for (int k = 0; k < 16; k++) {
        l[k] = Lk[i + k * DP];
        b[k] = i == k ? 1.0 : 0.0;
    }
    const double rd = rcp_nr(Lk[i + i * DP]);
    for_const<0, 16>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        b[k] *= row_value<k>(rd);
        for_const<k + 1, 16>([&](auto jc) {
            constexpr int j = decltype(jc)::value;
            b[j] = __builtin_fma(-b[k], row_value<j>(l[k]), b[j]);
        });
    });
    if (lane < 16) {
#pragma unroll
        for (int k = 0; k < 16; k++) Xk[k + i * DP] = b[k];
    }
}

// T_IJ = sum_{Q=J}^{I-1} L_IQ X_QJ (one wave): the off-diagonal block X_IJ of the inverse is -X_II T_IJ.
__device__ __forceinline__ d4_t tri_inv_sum(const double* D, const double* X, int I, int J) {
    d4_t T = {0, 0, 0, 0};
    for (int Q = J; Q < I; Q++) T = mma16(T, D + 16 * I + 16 * Q * DP, X + 16 * Q + 16 * J * DP, false);
    return T;
}
__device__ __forceinline__ void tri_inv_block(const double* D, double* X, int I, int J) {
    const d4_t T = tri_inv_sum(D, X, I, J);
    put16(X + 16 * I + 16 * J * DP, mma16_reg(X + 16 * I + 16 * I * DP, T), -1.0, false);
}
// Off-diagonal blocks of X = L^{-1} from L (D) and the diagonal inverses already in X, in order of I - J (one wave
// per block).
__device__ __forceinline__ void tri_inv_offdiag(const double* D, double* X) {
    const int wv = wave_uniform((int)threadIdx.x >> 6);
    for (int d = 1; d < 4; d++) {
        if (wv + d < 4) tri_inv_block(D, X, wv + d, wv);
        __syncthreads();
    }
}

// Factor D in place (lower; the upper part is left undefined) and write X = L^{-1}
// (lower, upper part zero); the LDS word after X is used too. Returns the first failing local column + 1 (0 if
// positive definite) to every thread.
// Four 16-column panels, each by wave 0 alone in registers (panel16): the chain of 64 pivots is what bounds this
// block, and a pivot step through LDS with a barrier takes ~0.25 us where one in registers takes ~0.1 us. The panel's
// spare lanes carry the identity, so the block's inverse comes out of the same pass; the other waves meanwhile do the
// updates that the next panel does not wait for and the off-diagonal blocks of the inverse. `beside` is run by wave 3
// while panel 0 is factored.
template <typename F>
__device__ __forceinline__ int lds_potrf_inv64(double* D, double* X, int w, const F& beside) {
    const int tid = threadIdx.x, lane = tid & 63, wv = wave_uniform(tid >> 6);
    int* s_bad = reinterpret_cast<int*>(X + DB * DP);
    if (tid == 0) *s_bad = 0;
    // D_IJ -= L_IK L_JK^T
    auto update = [&](int I, int J, int K) {
        const d4_t acc = mma16(d4_t{0, 0, 0, 0}, D + 16 * I + 16 * K * DP, D + 16 * J + 16 * K * DP, true);
        put16(D + 16 * I + 16 * J * DP, acc, -1.0, true);
    };
    d4_t T = {0, 0, 0, 0};
    __syncthreads();
#pragma unroll 1
    for (int K = 0; K < 4; K++) {
        const int k0 = 16 * K;
        // panel K: wave 0 holds rows k0 .. 63 and, in the lanes these leave, the identity; of panel 0 they leave none,
        // and wave 1 repeats the diagonal block with the identity below it
        if (wv == 0 || (wv == 1 && K == 0)) {
            const int nreal = wv == 0 ? DB - k0 : 16, e = lane - nreal;
            const int row = min(k0 + lane, DB - 1);
            double p[16], a[16];
#pragma unroll
            for (int c = 0; c < 16; c++) {
                p[c] = D[(k0 + (lane & 15)) + (k0 + c) * DP];
                a[c] = D[row + (k0 + c) * DP];
                if (lane >= nreal) a[c] = c == e ? 1.0 : 0.0;
            }
            if (K == 0) __syncthreads();  // both waves have read the block before wave 0 writes its factor
            const bool bad = panel16(p, a);
            if (wv == 0 && lane < nreal) {
#pragma unroll
                for (int c = 0; c < 16; c++) D[(k0 + lane) + (k0 + c) * DP] = a[c];
            } else if (e >= 0 && e < 16) {  // row e of L_KK^{-T}
#pragma unroll
                for (int c = 0; c < 16; c++) X[(k0 + c) + (k0 + e) * DP] = a[c];
            }
            if (wv == 0) {
                const unsigned long long m = __ballot(lane < 16 && k0 + lane < w && bad);
                if (m && lane == 0 && *s_bad == 0) *s_bad = k0 + __ffsll((long long)m);
            }
        } else if (K == 0) {  // waves 2, 3: the blocks above the diagonal of X
            for (int q = wv - 2; q < 6; q += 2) {
                const int J = q < 3 ? 3 : q < 5 ? 2 : 1, I = q < 3 ? q : q < 5 ? q - 3 : 0;
#pragma unroll
                for (int r = 0; r < 4; r++) X[16 * I + (lane & 15) + (16 * J + (lane >> 4) + 4 * r) * DP] = 0.0;
            }
            __syncthreads();
            if (wv == 3) beside();
        } else if (K == 1) {
            if (wv == 1) update(3, 2, 0);
            if (wv == 2) update(3, 3, 0);
        } else if (K == 3) {
            T = tri_inv_sum(D, X, 3, wv - 1);
        }
        __syncthreads();
        // what panel K + 1 waits for first
        if (K == 0) {
            if (wv < 3) update(1 + wv, 1, 0);
            else update(2, 2, 0);
        } else if (K == 1) {
            if (wv == 0) update(2, 2, 1);
            if (wv == 1) update(3, 2, 1);
            if (wv == 2) update(3, 3, 1);
            if (wv == 3) tri_inv_block(D, X, 1, 0);
        } else if (K == 2) {
            if (wv == 0) update(3, 3, 2);
            if (wv == 1) tri_inv_block(D, X, 2, 1);
            if (wv == 2) tri_inv_block(D, X, 2, 0);
        } else if (wv > 0) {
            put16(X + 48 + 16 * (wv - 1) * DP, mma16_reg(X + 48 + 48 * DP, T), -1.0, false);
        }
        __syncthreads();
    }
    return *s_bad;
}

// In-place style inverse of a lower-triangular 64x64 L held in D (w valid, identity
// padding set here): X = L^{-1}, lower, upper part zero.
__device__ __forceinline__ void lds_trtri64(double* D, double* X, int w) {
    const int tid = threadIdx.x, wv = wave_uniform(tid >> 6);
    for (int e = tid; e < DB * DB; e += NTHREADS) {
        const int i = e % DB, j = e / DB;
        if (i >= w || j >= w) D[i + j * DP] = (i == j) ? 1.0 : 0.0;
    }
    for (int e = tid; e < DB * DP; e += NTHREADS) X[e] = 0.0;
    __syncthreads();
    tri_inv16(D + 16 * wv + 16 * wv * DP, X + 16 * wv + 16 * wv * DP);
    __syncthreads();
    tri_inv_offdiag(D, X);
}

// Waits until *count >= want and returns the value seen. The polls are relaxed (an acquire
// load invalidates the L2 on every iteration, which with hundreds of waiting workgroups
// evicts everyone's data); one agent-scope acquire follows. Gives up after `limit` ticks
// (sets *err = 1) or as soon as *err is nonzero (an earlier wait timed out, or the owner
// asked the kernel to stop), so that a failed run drains in one time limit. `slow` polls
// about once a microsecond instead of back to back.
__device__ __forceinline__ int wait_count(const int32_t* count, int want, int32_t* err, int64_t limit,
                                          bool slow = false) {
    const int64_t t0 = (int64_t)wall_clock64();
    int v;
    while ((v = __hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) < want) {
        if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != 0) { v = want; break; }
        if ((int64_t)wall_clock64() - t0 > limit) {
            __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            v = want;
            break;
        }
        if (slow) __builtin_amdgcn_s_sleep(32);
        else __builtin_amdgcn_s_sleep(1);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    return v;
}


// ---------------------------------------------------------------------------
// POTRF of an n x n diagonal tile as items of 64x64 blocks, nb = ceil(n / 64) block rows (potrf_item): block items
// (r, q), q < r - 1, and per row a tail item, which owns blocks (r, r-1) and (r, r). An item keeps its
// blocks in registers and is left-looking:
//   A(r,q) -= L(r,j) L(q,j)^T, j = 0 .. q-1, each product once both blocks are published
//   L(r,q)  = A(r,q) X(q)^T once X(q) = L(q,q)^{-1} is published
// and the tail item also A(r,r) -= L(r,j) L(r,j)^T, j = 0 .. r-1, then factors and inverts the diagonal block in LDS
// and publishes X(r). Flag r (r + 1) / 2 + q says that L(r,q) (q < r) or X(r) (q = r) is final. Items are numbered row
// by row, so an item waits on lower-numbered items of its task only; these are claimed before it, and every wait ends.
// Why blocks and tails: the chain from X(r-1) to X(r) is one hand-over between workgroups, a triangular 64^3 product,
// the lower half of a 64^3 update and the diagonal block (8.8 us); everything else of row r has nb - r such steps
// to finish in. With one item per block row the last row's 35 products in series bounded a 512 tile (231 us).
// Outputs: L in the tile, the inverses in dinv. FP64 throughout; L is rounded to the tile's type as it is stored.
// ---------------------------------------------------------------------------
constexpr int BP = DB + 2;  // LDS pitch of a 64x64 operand block: Blk[k * BP + m] = element (m, k)
constexpr int LDS_POTRF = 2 * DB * BP * 8;
static_assert(DB * BP * 8 + DB * DP * 8 <= LDS_POTRF && (DB * DP + 1) * 8 <= DB * BP * 8, "D, X and its flag word fit");

// acc[cb] += At (rows 16w .. 16w+15) Bt^T (columns 16cb .. 16cb+15) of 64x64 operands in LDS; TRI: Bt is lower
// triangular (k <= column), its zero blocks are skipped. A lane's results: row 16w + l%16, columns 16cb + l/16 + 4r.
template <bool TRI>
__device__ __forceinline__ void mma64(d4_t (&acc)[4], const double* At, const double* Bt, int w) {
    const int lane = threadIdx.x & 63;
    const double* a0 = At + 16 * w + (lane & 15) + (lane >> 4) * BP;
    const double* b0 = Bt + (lane & 15) + (lane >> 4) * BP;
#pragma unroll
    for (int kb = 0; kb < 4; kb++)
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int k = 16 * kb + 4 * s;
            const double a = a0[k * BP];
#pragma unroll
            for (int cb = TRI ? kb : 0; cb < 4; cb++)
                acc[cb] = Mfma<double>::mma(b0[k * BP + 16 * cb], a, acc[cb]);
        }
}
// The lower 16x16 blocks (I, J) of a 64x64 block, shared out over four waves: three each to waves 0 and 1, two to
// waves 2 and 3. Nibble b of the code is I * 4 + J.
struct LowerBlocks {
    unsigned code;
    int cnt;
    __device__ __forceinline__ explicit LowerBlocks(int w)
        : code(w == 0 ? 0x0dcu : w == 1 ? 0x5feu : w == 2 ? 0x98u : 0x4au), cnt(w < 2 ? 3 : 2) {}
    __device__ __forceinline__ int I(int b) const { return (code >> (4 * b + 2)) & 3; }
    __device__ __forceinline__ int J(int b) const { return (code >> (4 * b)) & 3; }
};
// acc[b] += At At^T in this wave's lower blocks (a lane's results as in mma64).
__device__ __forceinline__ void mma64_lower(d4_t (&acc)[3], const double* At, const LowerBlocks& lb) {
    const int lane = threadIdx.x & 63;
    const double* a0 = At + (lane & 15) + (lane >> 4) * BP;
#pragma unroll
    for (int b = 0; b < 3; b++) {
        if (b < lb.cnt) {
            const double *pi = a0 + 16 * lb.I(b), *pj = a0 + 16 * lb.J(b);
#pragma unroll
            for (int ks = 0; ks < 16; ks++)
                acc[b] = Mfma<double>::mma(pj[4 * ks * BP], pi[4 * ks * BP], acc[b]);
        }
    }
}

// Two 64x64 blocks into LDS operand layout, every global load in flight before the first LDS store. Block P: element
// (m, k) at P[m + k * ldp], rows beyond `prows` zero; block Q whole.
template <typename TP, typename TQ>
__device__ __forceinline__ void stage_pair(double* At, const TTAD_GLOBAL TP* P, long ldp, int prows, double* Bt,
                                           const TTAD_GLOBAL TQ* Q, long ldq) {
    constexpr int PER = DB * DB / NTHREADS, KS = NTHREADS / DB;
    const int m = threadIdx.x % DB, k0 = threadIdx.x / DB;
    TP v[PER];
    TQ u[PER];
#pragma unroll
    for (int e = 0; e < PER; e++) {
        v[e] = P[min(m, prows - 1) + (long)(k0 + e * KS) * ldp];
        u[e] = Q[m + (long)(k0 + e * KS) * ldq];
    }
#pragma unroll
    for (int e = 0; e < PER; e++) {
        At[(k0 + e * KS) * BP + m] = m < prows ? (double)v[e] : 0.0;
        Bt[(k0 + e * KS) * BP + m] = (double)u[e];
    }
}
__device__ __forceinline__ void stage_inv(double* Bt, const TTAD_GLOBAL double* X) {
    constexpr int PER = DB * DB / NTHREADS, KS = NTHREADS / DB;
    const int m = threadIdx.x % DB, k0 = threadIdx.x / DB;
    double u[PER];
#pragma unroll
    for (int e = 0; e < PER; e++) u[e] = X[m + (k0 + e * KS) * DB];
#pragma unroll
    for (int e = 0; e < PER; e++) Bt[(k0 + e * KS) * BP + m] = u[e];
}

template <typename TS>
__device__ __forceinline__ void item_potrf(TS* __restrict__ A, long lda, int n, double* __restrict__ dinv, int* info,
                                           int col_off, int it, int32_t* flags, int32_t* err, int64_t spin_limit,
                                           char* lds) {
    const int tid = threadIdx.x, lane = tid & 63, w = wave_uniform(tid >> 6);
    const PotrfItem own = potrf_item(it);
    const int r = own.r, q = own.q;
    const bool tail = own.tail;
    const int p0 = r * DB, pw = min(DB, n - p0);
    auto flag = [&](int i, int j) { return flags + potrf_flag(i, j); };
    auto publish = [&](int i, int j) {
        release_agent();
        __hip_atomic_store(flag(i, j), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    double* At = reinterpret_cast<double*>(lds);
    double* Bt = At + DB * BP;
    TTAD_GLOBAL TS* Ag = gmem(A);
    TTAD_GLOBAL TS* Arow = Ag + p0;
    const int lr = 16 * w + (lane & 15), lc = lane >> 4;  // this lane's row of the block, first column of a fragment
    const LowerBlocks lb(w);
    // A(r, q) and the lower part of A(r, r), loaded ahead of the first wait; the sums of products are formed from
    // zero and subtracted once
    d4_t av[4], ad[3], acc[4], accd[3];
#pragma unroll
    for (int cb = 0; cb < 4; cb++) av[cb] = acc[cb] = d4_t{0, 0, 0, 0};
#pragma unroll
    for (int b = 0; b < 3; b++) ad[b] = accd[b] = d4_t{0, 0, 0, 0};
    if (r > 0) {
#pragma unroll
        for (int cb = 0; cb < 4; cb++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const double v = (double)Arow[min(lr, pw - 1) + (long)(q * DB + 16 * cb + lc + 4 * e) * lda];
                av[cb][e] = lr < pw ? v : 0.0;
            }
    }
    if (tail) {
#pragma unroll
        for (int b = 0; b < 3; b++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int rr = 16 * lb.I(b) + (lane & 15), cc = 16 * lb.J(b) + lc + 4 * e;
                const double v = (double)Arow[min(rr, pw - 1) + (long)(p0 + min(cc, pw - 1)) * lda];
                ad[b][e] = (rr < pw && cc < pw) ? v : (rr == cc ? 1.0 : 0.0);  // (identity padding)
            }
    }
    for (int j = 0; j < q; j++) {
        if (tid == 0) {
            wait_count(flag(r, j), 1, err, spin_limit);
            wait_count(flag(q, j), 1, err, spin_limit);
        }
        __syncthreads();  // both blocks are final; At / Bt are free
        stage_pair(At, Arow + (long)j * DB * lda, lda, pw, Bt, Ag + q * DB + (long)j * DB * lda, lda);
        __syncthreads();
        mma64<false>(acc, At, Bt, w);
        if (tail) mma64_lower(accd, At, lb);
    }
    if (r > 0) {
        __syncthreads();
#pragma unroll
        for (int cb = 0; cb < 4; cb++)
#pragma unroll
            for (int e = 0; e < 4; e++) At[(16 * cb + lc + 4 * e) * BP + lr] = av[cb][e] - acc[cb][e];
        if (tid == 0) wait_count(flag(q, q), 1, err, spin_limit);
        __syncthreads();
        stage_inv(Bt, gmem(dinv) + (long)q * DB * DB);
        __syncthreads();
#pragma unroll
        for (int cb = 0; cb < 4; cb++) acc[cb] = d4_t{0, 0, 0, 0};
        mma64<true>(acc, At, Bt, w);
        __syncthreads();
        // L(r, q) into the tile and, as stored, into LDS for the diagonal block's update
#pragma unroll
        for (int cb = 0; cb < 4; cb++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int cc = 16 * cb + lc + 4 * e;
                const TS v = (TS)acc[cb][e];
                if (lr < pw) Arow[lr + (long)(q * DB + cc) * lda] = v;
                At[cc * BP + lr] = (double)v;
            }
        if (tail) {
            __syncthreads();
            mma64_lower(accd, At, lb);
        }
        stores_done();
        if (!tail) {
            __syncthreads();
            if (tid == 0) publish(r, q);
        }
    }
    if (tail) {
        double *D = Bt, *X = At;
#pragma unroll
        for (int b = 0; b < 3; b++)
            if (b < lb.cnt) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int rr = 16 * lb.I(b) + (lane & 15), cc = 16 * lb.J(b) + lc + 4 * e;
                    D[rr + cc * DP] = ad[b][e] - accd[b][e];
                }
            }
        __syncthreads();
        const int bad = lds_potrf_inv64(D, X, pw, [&] {
            if (r > 0 && lane == 0) publish(r, q);  // its write-back runs beside the first panel
        });
        constexpr int PER = DB * DB / NTHREADS;
        const int i = tid % DB, j0 = tid / DB;
        TTAD_GLOBAL double* Xg = gmem(dinv) + (long)r * DB * DB;
#pragma unroll
        for (int e = 0; e < PER; e++) {
            const int j = j0 + e * (NTHREADS / DB);
            Xg[i + j * DB] = X[i + j * DP];
        }
        // (the word keeps the first report: a block that fails because of this one's NaNs waits for the flag below)
        if (bad && tid == 0) atomicCAS(info, 0, col_off + p0 + bad);
        stores_done();
        __syncthreads();
        if (tid == 0) publish(r, r);
#pragma unroll
        for (int e = 0; e < PER; e++) {
            const int j = j0 + e * (NTHREADS / DB);
            if (i < pw && j < pw && i >= j) Arow[i + (long)(p0 + j) * lda] = (TS)D[i + j * DP];
        }
    }
    if (tid == 0) {
        // the last item of the task to finish clears the flags for the next run on this tile; every item's own flags have
        // arrived by then, since it waits for these stores before it counts itself
        stores_done();
        if (__hip_atomic_fetch_add(flags + potrf_fin(n), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == potrf_items(n) - 1)
            for (int e = 0; e < potrf_flags(n); e++)
                __hip_atomic_store(flags + e, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// ---------------------------------------------------------------------------
// TRSM work item: trsm_rows(sizeof(TS), false) rows of X (m x n) := X L^{-T} (Right, Lower,
// Trans, NonUnit), in place, by 64-column blocks: the block's right-hand side goes
// into the accumulators, the already solved columns times L's off-diagonal blocks
// are subtracted (one GEMM), and the result is multiplied by the inverse of L's
// 64x64 diagonal block left by POTRF straight from LDS (no round trip through
// memory between the two products). TC is the MFMA type (FP64, or FP32 for the
// mixed variants).
// ---------------------------------------------------------------------------
// planes (FP32 tiles; null = none): the bf16 split planes of X (ldx rows, plane_granule layout), written
// beside X for the bf16x3 updates that read it; needs n % 32 == 0.
template <typename TS, typename TC>
__device__ __forceinline__ void item_trsm(const TS* __restrict__ L, long ldl, const double* __restrict__ dinv, TS* __restrict__ X,
                          long ldx, int m, int n, int r0, char* lds, void* planes = nullptr) {
    constexpr bool VEC = std::is_same<TS, TC>::value;
    constexpr int BMT = trsm_rows(sizeof(TS), false);
    using G = GemmNT<TS, TS, TC, BMT, DB, trsm_bk<TS>(), VEC, true>;  // update from the solved columns
    using G3 = GemmNT<TC, TC, TC, BMT, DB, DB, false, true>;  // times Dinv^T, both operands in LDS
    const int mv = min(BMT, m - r0);
    if (mv <= 0) return;
    TS* Xr = X + r0;
    const int nblk = (n + DB - 1) / DB;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, wr = w >> 1, wc = w & 1;
    TC* At = reinterpret_cast<TC*>(lds);  // G3 staging: At[k][m] = t(m, k), Bt[k][j] = Dinv(j, k)
    TC* Bt = At + DB * G3::PA;
    typename G::acc_t acc[G::WM][G::WN];
    for (int cb = 0; cb < nblk; cb++) {
        const int c0 = cb * DB, cw = min(DB, n - c0);
        TTAD_GLOBAL TS* T = gmem(Xr) + (long)c0 * ldx;
        // acc = -(right-hand side block) + X[:, :c0] L[c0:c0+cw, :c0]^T = -t
#pragma unroll
        for (int a = 0; a < G::WM; a++)
#pragma unroll
            for (int b = 0; b < G::WN; b++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int rr = G::row_of(a, r), cc = G::col_of(b, r);
                    acc[a][b][r] = (rr < mv && cc < cw) ? -(TC)T[rr + (long)cc * ldx] : TC(0);
                }
        if (c0 > 0) G::run(acc, Xr, ldx, mv, L + c0, ldl, cw, c0, lds);
        else __syncthreads();  // the previous block's products have left the staging area
#pragma unroll
        for (int a = 0; a < G::WM; a++)
#pragma unroll
            for (int b = 0; b < G::WN; b++)
#pragma unroll
                for (int r = 0; r < 4; r++) At[G::col_of(b, r) * G3::PA + G::row_of(a, r)] = -acc[a][b][r];
        // Dinv block into Bt, every global load in flight before the first LDS store (a
        // load-store loop would wait for each load in turn)
        {
            constexpr int PER = DB * DB / (2 * NTHREADS);
            using d2 = V16<double>::t;
            const TTAD_GLOBAL d2* Dv = reinterpret_cast<const TTAD_GLOBAL d2*>(gmem(dinv) + (long)cb * DB * DB);
            d2 v[PER];  // Dv[i + j*DB] = Dinv(i, j), two rows of a column per element
#pragma unroll
            for (int q = 0; q < PER; q++) v[q] = Dv[threadIdx.x + q * NTHREADS];
#pragma unroll
            for (int q = 0; q < PER; q++) {
                const int e = 2 * (threadIdx.x + q * NTHREADS);
                TC* d = Bt + (e / DB) * G3::PB + (e % DB);
                d[0] = (TC)v[q].x;
                d[1] = (TC)v[q].y;
            }
        }
        __syncthreads();
        G3::zero(acc);
        G3::compute(acc, At, lane, wr, wc);
#pragma unroll
        for (int a = 0; a < G::WM; a++)
#pragma unroll
            for (int b = 0; b < G::WN; b++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int rr = G3::row_of(a, r), cc = G3::col_of(b, r);
                    if (rr < mv && cc < cw) T[rr + (long)cc * ldx] = (TS)acc[a][b][r];
                }
        if constexpr (std::is_same<TS, float>::value && std::is_same<TC, float>::value) {
            // a lane holds 4 consecutive columns of one row per fragment (cw is a multiple of 32 here)
            if (planes) {
#pragma unroll
                for (int a = 0; a < G::WM; a++)
#pragma unroll
                    for (int b = 0; b < G::WN; b++) {
                        const int rr = G3::row_of(a, 0), cc = G3::col_of(b, 0);
                        if (rr < mv && cc < cw)
                            store_split4(static_cast<unsigned short*>(planes), (int)ldx, r0 + rr, c0 + cc, acc[a][b]);
                    }
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// TRSM work item for n <= TRSM_LDS_COLS columns: trsm_rows(sizeof(TS), true) rows of X := X L^{-T}, in place. The solved
// columns stay in LDS (Xs[k][m]), where the next columns' products read them; L's blocks go from the L2 straight into
// MFMA operands (a lane's element L(c, k), 128-byte segments), three chunks of 64 columns ahead: they do not depend on
// the solve, so the loads run through its serial steps. Per 64-column block: wave w forms columns 16w .. 16w+15 of
//   -t = -rhs + Xs L(block, 0:c0)^T, exchanged through LDS, then x = t Dinv^T (Dinv lower triangular)
// with two barriers; sums in the order of item_trsm, so both forms give the same bits. What bounds it: the MFMAs of one
// strip (512 columns in FP64: 12 us) and the exchanges. 256 columns 31 -> 17 us, 512 columns 90 -> 42 us (FP64, idle CUs).
// Which TRSM tasks take it: the strip is half as high as item_trsm's, so L is read twice as often; FP32 tasks gain at
// every size (bf16x3 n = 16384: 10.8 -> 9.0 ms), FP64 ones while the chain bounds the run (graph_prepare).
// ---------------------------------------------------------------------------
constexpr int TRSM_RING = 3;  // chunks of L in flight
template <typename TS>
__device__ __forceinline__ void item_trsm_lds(const TS* __restrict__ L, long ldl, const double* __restrict__ dinv,
                                              TS* __restrict__ X, long ldx, int m, int n, int r0, char* lds,
                                              void* planes = nullptr) {
    typedef Mfma<TS> MF;
    typedef typename MF::acc_t acc_t;
    constexpr int RM = trsm_rows(sizeof(TS), true), RB = RM / 16;  // rows of the item, 16-row blocks
    const int mv = min(RM, m - r0);
    if (mv <= 0) return;
    TS* Xs = reinterpret_cast<TS*>(lds);     // Xs[k * RM + m]
    TS* Ts = Xs + TRSM_LDS_COLS * RM;        // the exchanged block, Ts[k * RM + m]
    const int lane = threadIdx.x & 63, w = wave_uniform((int)threadIdx.x >> 6), l15 = lane & 15, kl = lane >> 4;
    const int nblk = (n + DB - 1) / DB;
    TTAD_GLOBAL TS* Xg = gmem(X) + r0;
    TS bq[TRSM_RING][16];
    // Element `off` bytes behind a uniform pointer: a scalar base and a 32-bit lane offset, no 64-bit lane address per
    // load (trsm_lane_offset).
    auto at = [](auto* base, unsigned off) {
        using T = typename std::remove_cv<typename std::remove_pointer<decltype(base)>::type>::type;
        return *reinterpret_cast<const TTAD_GLOBAL T*>(reinterpret_cast<const TTAD_GLOBAL char*>(gmem(base)) + off);
    };
    const unsigned lds_k = (unsigned)kl * (unsigned)ldl;  // this lane's k offset in L
    // chunk kc of block cb into ring slot q: lane's elements L(64 cb + 16 w + l15, 64 kc + 4 ks + kl)
    auto fetch = [&](TS (&b)[16], int cb, int kc) {
        const unsigned off = ((unsigned)min(cb * DB + 16 * w + l15, n - 1) + lds_k) * (unsigned)sizeof(TS);
#pragma unroll
        for (int ks = 0; ks < 16; ks++) b[ks] = at(L + (long)(kc * DB + 4 * ks) * ldl, off);
    };
    auto fetch_block = [&](int cb) {
#pragma unroll
        for (int q = 0; q < TRSM_RING; q++)
            if (q < cb) fetch(bq[q], cb, q);
    };
    TS rhs[RB][4];  // the right-hand side block of the next column block (result layout)
    auto fetch_rhs = [&](int cb) {
        const int c0 = cb * DB, cw = min(DB, n - c0);
        const TS* base = X + r0 + (long)(c0 + trsm_wave_col(w, cw)) * ldx;
#pragma unroll
        for (int a = 0; a < RB; a++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                rhs[a][r] = at(base, trsm_lane_offset(min(16 * a + l15, mv - 1), MF::row(lane, r), w, cw, ldx, sizeof(TS)));
    };
    fetch_rhs(0);
    for (int cb = 0; cb < nblk; cb++) {
        const int c0 = cb * DB, cw = min(DB, n - c0);
        double dv[16];  // Dinv(16 w + l15, 4 ks + kl); zero above the diagonal
#pragma unroll
        for (int ks = 0; ks < 16; ks++)
            dv[ks] = at(dinv + (long)cb * DB * DB + 4 * ks * DB, (unsigned)(16 * w + l15 + kl * DB) * 8u);
        acc_t acc[RB];
#pragma unroll
        for (int a = 0; a < RB; a++) acc[a] = acc_t{-rhs[a][0], -rhs[a][1], -rhs[a][2], -rhs[a][3]};
        if (cb + 1 < nblk) fetch_rhs(cb + 1);
        auto product = [&](const TS (&b)[16], const TS* A) {
#pragma unroll
            for (int ks = 0; ks < 16; ks++)
#pragma unroll
                for (int a = 0; a < RB; a++)
                    acc[a] = MF::mma(b[ks], A[(4 * ks + kl) * RM + 16 * a + l15], acc[a]);
        };
        for (int kc = 0; kc < cb; kc += TRSM_RING)
#pragma unroll
            for (int q = 0; q < TRSM_RING; q++)
                if (kc + q < cb) {
                    product(bq[q], Xs + (kc + q) * DB * RM);
                    if (kc + q + TRSM_RING < cb) fetch(bq[q], cb, kc + q + TRSM_RING);
                }
        if (cb + 1 < nblk) fetch_block(cb + 1);
#pragma unroll
        for (int a = 0; a < RB; a++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                Ts[(16 * w + MF::row(lane, r)) * RM + 16 * a + l15] = -acc[a][r];
        __syncthreads();
#pragma unroll
        for (int a = 0; a < RB; a++) acc[a] = acc_t{0, 0, 0, 0};
        TS db[16];
#pragma unroll
        for (int ks = 0; ks < 16; ks++) db[ks] = (TS)dv[ks];
#pragma unroll
        for (int ks = 0; ks < 16; ks++)
            if (ks < 4 * (w + 1)) {
#pragma unroll
                for (int a = 0; a < RB; a++)
                    acc[a] = MF::mma(db[ks], Ts[(4 * ks + kl) * RM + 16 * a + l15], acc[a]);
            }
#pragma unroll
        for (int a = 0; a < RB; a++) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int cc = 16 * w + MF::row(lane, r);
                Xs[(c0 + cc) * RM + 16 * a + l15] = acc[a][r];
                if (16 * a + l15 < mv && cc < cw) Xg[16 * a + l15 + (long)(c0 + cc) * ldx] = acc[a][r];
            }
            if constexpr (std::is_same<TS, float>::value) {
                // a lane holds 4 consecutive columns of one row (cw is a multiple of 32 where there are planes)
                const int cc = 16 * w + MF::row(lane, 0);
                if (planes && 16 * a + l15 < mv && cc < cw)
                    store_split4(static_cast<unsigned short*>(planes), (int)ldx, r0 + 16 * a + l15, c0 + cc, acc[a]);
            }
        }
        __syncthreads();
    }
}

template <typename TS> constexpr int trsm_lds_bytes() {
    return (TRSM_LDS_COLS + DB) * trsm_rows(sizeof(TS), true) * (int)sizeof(TS);
}

// LDS bytes each item kind needs (the executor reserves the maximum).
constexpr int LDS_GEMM_F64 = GemmNT<double, double, double, GEMM_BM, GEMM_BM, gemm_bk<double>(), true, true>::LDS_BYTES;
constexpr int LDS_GEMM_F32 = GemmNT<float, float, float, GEMM_BM, GEMM_BM, gemm_bk<float>(), true, true>::LDS_BYTES;
constexpr int LDS_GEMM_BF16 = GemmNTbf16<float, GEMM_BM, GEMM_BM, true, true>::LDS_BYTES;
constexpr int LDS_GEMM_BF16_1 = GemmNTbf16<float, GEMM_BM, GEMM_BM, false, true>::LDS_BYTES;
// LDS of one GEMM item of the given storage / precision (the standalone kernels launch with it).
template <typename TS, int PREC, int BM = GEMM_BM> constexpr int gemm_item_lds() {
    if (BM != GEMM_BM)
        return PREC == P_BF16X3 ? GemmNTbf16<float, BM, BM, true, true>::LDS_BYTES
               : PREC == P_BF16 ? GemmNTbf16<float, BM, BM, false, true>::LDS_BYTES
                                : GemmNT<TS, TS, TS, BM, BM, gemm_bk<TS, BM>(), true, true>::LDS_BYTES;
    return PREC == P_BF16X3 ? LDS_GEMM_BF16 : PREC == P_BF16 ? LDS_GEMM_BF16_1 : sizeof(TS) == 8 ? LDS_GEMM_F64 : LDS_GEMM_F32;
}
constexpr int LDS_TRSM = cmax(GemmNT<double, double, double, TRSM_BM, DB, 32, true, true>::LDS_BYTES,
                              GemmNT<double, double, double, TRSM_BM, DB, DB, false, true>::STAGE * 8);
constexpr int LDS_TRSM_F32 = cmax(GemmNT<float, float, float, TRSM_BM_F32, DB, trsm_bk<float>(), true, true>::LDS_BYTES,
                                  GemmNT<float, float, float, TRSM_BM_F32, DB, DB, false, true>::STAGE * 4);
constexpr int LDS_ITEM_MAX =
    cmax(cmax(cmax(LDS_GEMM_F64, LDS_GEMM_F32), cmax(LDS_GEMM_BF16, LDS_POTRF)),
         cmax(LDS_TRSM, cmax(trsm_lds_bytes<double>(), trsm_lds_bytes<float>())));

}  // namespace ttad
