// Block-sparse S stage of the grouped sigma / boundary steps on gfx950 MFMA:
//
//   S_D[:, panel] = T_D[:, K runs] * W_D[K runs, panel]      per charge-transfer group D
//
// W_D's keys are in pattern-class order (engine.hip, reorder_group_keys), so its nonzeros sit in
// dense rectangles; every 128-column panel of W_D keeps only its 16-key tiles that hold a nonzero,
// stored compactly ([n][16 k] per tile, zero padded) and grouped into runs of consecutive tiles.
// One workgroup computes one 128 x 128 tile of S_D: it walks the runs of its panel, reading the
// T_D rows (column-major, rows contiguous) straight into registers in the MFMA layout, since every wave
// has rows of its own, and the compact W tiles, which all waves share, through LDS, double buffered.
//
// What bounds it: FP64 the MFMA rate (matrix units busy 80% of the time; 61 of the 73 TFLOP/s a large FP64
// product reaches, counting the zeros inside visited 16 x 16 blocks), BF16X3 the memory: at L=30, m=1500
// it reads 31 GB and writes 8.4 GB in 8.3 ms, 4.8 TB/s, where T_D once is 8.2 GB.  The 8 x 8 panel blocks ask
// for T_D once per 8 column panels and for W once per 8 row panels, 18 and 5 GB; the rest of what is read
// comes back because a block's panels do not stay in L2 for all of it.  A visited 16 x 128 tile is on average
// two thirds full by 16-column blocks; every wave spans the tile's 128 columns and skips the blocks without
// a nonzero (the same for every wave; adding a zero product of finite values changes no bit), and the loads
// run two steps ahead.  S stage at SU2U1 L=30 m=1500: FP64
// 49.8 ms with every block multiplied, 30.8 ms with blocks skipped, tiles dealt to the XCDs and T_D staged
// through LDS, 26.1 ms with T_D read directly, W read in whole lines and 8 waves; BF16X3 9.3 -> 8.3 ms.
// L=24 m=1000: FP64 13.3, 7.1, 5.8 ms; BF16X3 2.85, 2.45, 2.2 ms.  Three arithmetics:
//
//   MODE_F64     v_mfma_f64_16x16x4f64 on FP64 T_D / W tiles (the plain path)
//   MODE_F32     v_mfma_f32_16x16x4f32 on FP32 T_D / W tiles
//   MODE_BF16X3  FP32 T_D split on the fly into bf16 hi + lo in registers, W tiles split once
//                per plan; three v_mfma_f32_16x16x32_bf16 products per block and 32-key step
//                (hi*lo + lo*hi + hi*hi) with FP32 accumulation, the split-product scheme of the
//                library path (gfx950's K = 32 bf16 MFMA: twice the rate per key of the K = 16 form)
//
// The reference's S stage is a gather over the nonzero MPO couplings alpha
// (solver/numeric/gpu_dgemm_ddot.cu:282-359, solver/tasks.cpp:466-504); here the couplings of one
// group form W_D and its empty tiles are never visited.  Each output element is written once, by
// one workgroup, with a fixed summation order: the stage is deterministic.
//
// MFMA lane layouts (lane l, lk = l / 16):
//   f64 16x16x4        A row l%16, k lk;  B col l%16, k lk;  D[r] row 4r + lk, col l%16
//   f32 16x16x4        A row l%16, k lk;  B col l%16, k lk;  D[r] row 4lk + r, col l%16
//   bf16 16x16x32      A row l%16, 8 k per lane;  B col l%16, the same 8 k;  D[r] row 4lk + r
// (the bf16 kernel gives lane group lk the keys 8 lk .. 8 lk + 7 of its row and of its column; the
// sum over k does not depend on which of the 32 k positions each key takes, as long as A and B
// agree, and they use one layout)
#include <hip/hip_runtime.h>

#include <type_traits>

#include "kernels.hpp"

namespace mq {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

constexpr int BM = S_BSR_TILE_M, BN = S_BSR_TILE_N, BK = S_BSR_TILE_K;
static_assert(BM == 128 && BN == 128 && BK == 16, "tile shape");

// Two elements: hi = bf16(x), lo = bf16(x - hi), round to nearest even (the rule of bf16_rne, the T
// stage's split), each pair packed with the lower element in the low half.  The float -> bf16
// conversions are gfx950's v_cvt_pk_bf16_f32 (two values per instruction).
__device__ inline void split_bf16x2(float x0, float x1, uint32_t& hi, uint32_t& lo) {
    hi = __builtin_bit_cast(uint32_t, bf2{(__bf16)x0, (__bf16)x1});
    asm("" : "+v"(hi));   // one conversion for both: the halves below are taken from the pair
    const float h0 = __uint_as_float(hi << 16), h1 = __uint_as_float(hi & 0xffff0000u);
    lo = __builtin_bit_cast(uint32_t, bf2{(__bf16)(x0 - h0), (__bf16)(x1 - h1)});
}

// A load at base + uniform + lane byte offset (base and uniform the same for the wave), 0 if the two offsets
// reach `bytes`: buffer loads take them as they are, so that a step's loads cost no address arithmetic,
// no address registers and no branch at a run's end.
template <class V>
__device__ inline V buf_load(const void* base, uint32_t bytes, uint32_t uniform, uint32_t lane) {
    __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, int(bytes), 0x00020000);
    if constexpr (sizeof(V) == 16)
        return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(r, lane, uniform, 0));
    else
        return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(r, lane, uniform, 0));
}

template <int MODE> struct BsrTraits;
template <> struct BsrTraits<MODE_F64> { typedef double T; typedef d4 Acc; };
template <> struct BsrTraits<MODE_F32> { typedef float T; typedef f4 Acc; };
template <> struct BsrTraits<MODE_BF16X3> { typedef float T; typedef f4 Acc; };

// One step's W tiles in LDS, [n][k].  FP64 / FP32 rows are padded by 16 bytes: 16-byte chunks are stored
// whole.  FP64's reads meet banks twice at that stride (45% of the LDS cycles); rows of 17 doubles, read
// without a conflict but stored by halves, were slower (L=30 m=1500: 27.1 against 26.4 ms).  BF16X3: rows of 32 keys, 16-byte
// chunks of 8 keys, chunk c of row n at c ^ (n / 2 % 4): 8 lanes that read (or store) the same chunk of 8
// consecutive rows meet 8 different chunks of the 32 banks (no conflict counted).
template <int MODE> struct BsrSmem {
    typedef typename BsrTraits<MODE>::T T;
    T b[BN][BK + 16 / sizeof(T)];
};
template <> struct BsrSmem<MODE_BF16X3> {
    uint16_t bhi[BN][2 * BK], blo[BN][2 * BK];
    __device__ static int at(int n, int chunk) { return (chunk ^ (n >> 1 & 3)) * 8; }
};
// BF16X3 steps over two 16-key tiles (32 keys): its MFMAs are 16x faster per key than FP32's, and
// one tile per step left too little work between two waits on global memory.  WI 16-row blocks per
// wave: FP64 takes 8 waves of 16 x 128 (128 registers, 4 waves per SIMD), the others 4 of 32 x 128.
template <int MODE> struct BsrStep { static constexpr int KS = BK, WI = MODE == MODE_F64 ? 1 : 2, NT = 64 * BM / (16 * WI); };
template <> struct BsrStep<MODE_BF16X3> { static constexpr int KS = 2 * BK, WI = 2, NT = 256; };

template <int MODE, bool NARROW>
__global__ __launch_bounds__(BsrStep<MODE>::NT) __attribute__((amdgpu_waves_per_eu(MODE == MODE_F64 ? 4 : MODE == MODE_F32 ? 3 : 2))) void s_bsr_kernel(
    const BsrTask* __restrict__ tasks, const BsrRun* __restrict__ runs, const uint32_t* __restrict__ tile_cols,
    const void* __restrict__ bt0, const void* __restrict__ bt1, void* __restrict__ ws) {
    typedef typename BsrTraits<MODE>::T T;
    typedef typename BsrTraits<MODE>::Acc Acc;
    typedef BsrStep<MODE> Step;
    constexpr bool BF = MODE == MODE_BF16X3;
    constexpr int NT = Step::NT, KS = Step::KS, WI = Step::WI, WJ = BN / 16;
    __shared__ __align__(16) BsrSmem<MODE> sm[2];

    // a block of 8 x 8 panels of one group (64 tasks) runs on one XCD; the blocks are dealt to the XCDs in turn
    const uint32_t tile = xcd_tile_cyclic<64>(blockIdx.x, gridDim.x);
    const BsrTask tk = tasks[tile];
    const T* __restrict__ A = reinterpret_cast<const T*>(ws) + tk.a_off;
    T* __restrict__ C = reinterpret_cast<T*>(ws) + tk.c_off;
    const uint32_t M = tk.M, N = tk.N;
    const uint64_t ld = tk.ld;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, lk = lane >> 4;
    const int row0 = (wave * 16 + l16) * WI;   // the lane's rows row0 .. row0 + WI - 1, one per 16-row block

    Acc acc[WI][WJ];
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
        for (int j = 0; j < WJ; ++j) acc[i][j] = Acc{0, 0, 0, 0};

    // ---- loads of one step of KS keys (run r, key offset kk within the run)
    // A: every wave reads its own T_D rows straight into the MFMA layout, 16 lanes consecutive rows of one
    // key column (128 bytes); load e takes the keys KE e + KL lk.  Rows beyond M read valid workspace
    // memory (the plan checks 128 rows past every panel); they only feed output rows that are not
    // stored.  Keys beyond the run's end read as zero (buffer loads) or as its last key: their W
    // entries are zero (the run's last tile is zero padded, and a tile past the run's end counts as
    // zero), so they add nothing.  NARROW, (KS * ld + BM) elements of every task fit in 2^32 bytes: 32-bit
    // lane offsets, and buffer loads where that is faster (FP64 L=30: 26.9 -> 26.1 ms; BF16X3 8.3 -> 8.5 ms,
    // so it keeps pointers).
    // B: the compact tile(s) (128 columns x 16 keys each, [n][k]) in 16-byte chunks, consecutive lanes
    // (BF16X3: 16 lanes) read consecutive chunks; BF16X3 one chunk of each half of the split per tile.
    constexpr int AK = BF ? 8 : BK / 4, KE = BF ? 1 : 4, KL = BF ? 8 : 1;
    typedef T __attribute__((ext_vector_type(WI), aligned(sizeof(T)))) VA;
    constexpr int CW = 16 / (BF ? 2 : int(sizeof(T))), CN = BK / CW;   // keys per chunk, chunks per column
    constexpr int BV = BF ? 4 : BN * CN / NT;                          // chunks per thread
    const int b_n = BF ? (tid >> 4) * 8 + (tid & 7) : tid / CN, b_c = BF ? tid >> 3 & 1 : tid % CN;
    const uint32_t b_off = uint32_t(b_n * CN + b_c) * 16;
    typedef typename std::conditional<NARROW, uint32_t, uint64_t>::type Off;
    const Off ld_b = Off(ld) * Off(sizeof(T));
    const Off a_row = Off(row0) * Off(sizeof(T)), a_off = a_row + Off(KL * lk) * ld_b;
    struct Stage {
        VA va[AK];
        uint4 vb[BV];
        uint32_t cols;   // 16-column blocks of the step with a nonzero
        bool two;        // BF16X3: the step's second tile is within the run
    };
    auto fetch = [&](Stage& g, const BsrRun& R, uint32_t kk) {
        const uint32_t t = R.tile + kk / BK;
        g.cols = tile_cols[t];
        if constexpr (BF) {
            g.two = kk + BK < R.nk;
            const uint32_t t2 = t + g.two;
            g.cols |= tile_cols[t2];
            const uint16_t* hi = reinterpret_cast<const uint16_t*>(bt0);
            const uint16_t* lo = reinterpret_cast<const uint16_t*>(bt1);
            const char* p[4] = {reinterpret_cast<const char*>(hi + uint64_t(t) * (BN * BK)),
                                reinterpret_cast<const char*>(lo + uint64_t(t) * (BN * BK)),
                                reinterpret_cast<const char*>(hi + uint64_t(t2) * (BN * BK)),
                                reinterpret_cast<const char*>(lo + uint64_t(t2) * (BN * BK))};
#pragma unroll
            for (int v = 0; v < 4; ++v) g.vb[v] = *reinterpret_cast<const uint4*>(p[v] + b_off);
        } else {
            const char* p = reinterpret_cast<const char*>(reinterpret_cast<const T*>(bt0) + uint64_t(t) * (BN * BK));
#pragma unroll
            for (int v = 0; v < BV; ++v) g.vb[v] = buf_load<uint4>(p, BN * BK * sizeof(T), v * NT * 16, b_off);
        }
        const char* col = reinterpret_cast<const char*>(A + (uint64_t(R.k0) + kk) * ld);   // the step's first key column
        if constexpr (NARROW && !BF) {
            const uint32_t bytes = min(R.nk - kk, uint32_t(KS)) * ld_b;
#pragma unroll
            for (int e = 0; e < AK; ++e) g.va[e] = buf_load<VA>(col, bytes, uint32_t(e * KE) * ld_b, a_off);
        } else if (kk + KS <= R.nk) {
#pragma unroll
            for (int e = 0; e < AK; ++e)
                g.va[e] = *reinterpret_cast<const VA*>(col + uint64_t(e * KE) * (ld * sizeof(T)) + a_off);
        } else {
            const uint32_t last = R.nk - 1 - kk;   // last key of the run, relative to the step
#pragma unroll
            for (int e = 0; e < AK; ++e)
                g.va[e] = *reinterpret_cast<const VA*>(col + (a_row + Off(min(uint32_t(KE * e + KL * lk), last)) * ld_b));
        }
    };
    auto lstore = [&](const Stage& g, int buf) {
        BsrSmem<MODE>& s = sm[buf];
        if constexpr (BF) {
            *reinterpret_cast<uint4*>(&s.bhi[b_n][s.at(b_n, b_c)]) = g.vb[0];
            *reinterpret_cast<uint4*>(&s.blo[b_n][s.at(b_n, b_c)]) = g.vb[1];
            *reinterpret_cast<uint4*>(&s.bhi[b_n][s.at(b_n, b_c + 2)]) = g.two ? g.vb[2] : uint4{0, 0, 0, 0};
            *reinterpret_cast<uint4*>(&s.blo[b_n][s.at(b_n, b_c + 2)]) = g.two ? g.vb[3] : uint4{0, 0, 0, 0};
        } else {
#pragma unroll
            for (int v = 0; v < BV; ++v) *reinterpret_cast<uint4*>(&s.b[b_n + v * (NT / CN)][b_c * CW]) = g.vb[v];
        }
    };
    // the step's T_D operands: as loaded, or split
    struct Frag {
        T a[BF ? 1 : WI][BF ? 1 : AK];
        uint4 hi[WI], lo[WI];
    };
    auto take = [&](const Stage& g) {
        Frag f;
#pragma unroll
        for (int i = 0; i < WI; ++i) {
            if constexpr (BF) {
                uint32_t h[4], l[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) split_bf16x2(g.va[2 * e][i], g.va[2 * e + 1][i], h[e], l[e]);
                f.hi[i] = uint4{h[0], h[1], h[2], h[3]};
                f.lo[i] = uint4{l[0], l[1], l[2], l[3]};
            } else {
#pragma unroll
                for (int e = 0; e < AK; ++e) f.a[i][e] = g.va[e][i];
            }
        }
        return f;
    };
    // acc^T += W^T T_D^T: the columns of S_D are the MFMA's rows
    auto compute = [&](int buf, const Frag& f, uint32_t cols) {
        const BsrSmem<MODE>& s = sm[buf];
        if constexpr (BF) {
            // a block's W operands are read while the one before is multiplied
            bf8 bh[2], bl[2];
            auto read = [&](int j) {
                const int n = 16 * j + l16;
                bh[j & 1] = *reinterpret_cast<const bf8*>(&s.bhi[n][s.at(n, lk)]);
                bl[j & 1] = *reinterpret_cast<const bf8*>(&s.blo[n][s.at(n, lk)]);
            };
            read(0);
#pragma unroll
            for (int j = 0; j < WJ; ++j) {
                if (j + 1 < WJ) read(j + 1);
                if (!(cols >> j & 1)) continue;   // uniform: the step's 16 columns are all zero
#pragma unroll
                for (int i = 0; i < WI; ++i) {
                    const bf8 ah = __builtin_bit_cast(bf8, f.hi[i]), al = __builtin_bit_cast(bf8, f.lo[i]);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bl[j & 1], ah, acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[j & 1], al, acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[j & 1], ah, acc[i][j], 0, 0, 0);
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < WJ; ++j) {
                if (!(cols >> j & 1)) continue;   // uniform: the step's 16 columns are all zero
                const int n = 16 * j + l16;
                T b[AK];
#pragma unroll
                for (int e = 0; e < AK; ++e) b[e] = s.b[n][4 * e + lk];
#pragma unroll
                for (int e = 0; e < AK; ++e)
#pragma unroll
                    for (int i = 0; i < WI; ++i) {
                        if constexpr (MODE == MODE_F64)
                            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[e], f.a[i][e], acc[i][j], 0, 0, 0);
                        else
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[e], f.a[i][e], acc[i][j], 0, 0, 0);
                    }
            }
        }
    };

    // ---- the steps of all runs of the panel.  While step t is computed, step t + 1 waits in registers
    // (its W tiles go to the other LDS buffer after the products) and step t + 2's loads are issued: two
    // steps of work cover a load's latency.
    // Past the last step the loads repeat it (unused): every path through the loop issues the same
    // loads, so the wait before a store counts only the older step's.
    uint32_t r = tk.run0, kk = 0;
    if (r < tk.run1) {
        const uint32_t last_run = tk.run1 - 1;
        BsrRun R = runs[r], Rn = runs[min(r + 1, last_run)];   // the next run is at hand before it is needed
        auto advance = [&]() -> uint32_t {   // to the next step; 0 (and stays) at the last
            if (kk + KS < R.nk) {
                kk += KS;
                return 1;
            }
            if (r == last_run) return 0;
            R = Rn;
            ++r;
            Rn = runs[min(r + 1, last_run)];
            kk = 0;
            return 1;
        };
        Stage ga, gb;
        fetch(ga, R, kk);
        uint32_t has = advance();
        fetch(gb, R, kk);
        lstore(ga, 0);
        __syncthreads();
        // two steps a turn and one way out: the second of an odd last turn repeats loads and multiplies
        // nothing (a way out between them would make the compiler wait for the newest loads)
        uint32_t more;
        do {
            {
                const Frag f = take(ga);
                const uint32_t cols = ga.cols;
                more = has ? advance() : 0;
                fetch(ga, R, kk);
                compute(0, f, cols);
                lstore(gb, 1);
                __syncthreads();
            }
            {
                const Frag f = take(gb);
                const uint32_t cols = has ? gb.cols : 0;
                has = more ? advance() : 0;
                fetch(gb, R, kk);
                compute(1, f, cols);
                lstore(ga, 0);
                __syncthreads();
            }
        } while (more);
    }

    // ---- epilogue: C = acc (rows < M, columns < N).  A lane holds 4 columns of its rows: a store
    // instruction 128 bytes along the rows of 4 columns (element-aligned vector stores are legal for
    // global memory)
#pragma unroll
    for (int j = 0; j < WJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t col = 16 * j + (MODE == MODE_F64 ? 4 * q + lk : 4 * lk + q);
            if (col >= N || uint32_t(row0) >= M) continue;
            T* cc = C + uint64_t(col) * ld + row0;
            if constexpr (WI == 2) {
                if (uint32_t(row0) + 1 < M)
                    *reinterpret_cast<VA*>(cc) = VA{acc[0][j][q], acc[1][j][q]};
                else
                    cc[0] = acc[0][j][q];
            } else {
                cc[0] = acc[0][j][q];
            }
        }
}

}  // namespace

hipError_t launch_s_bsr(hipStream_t st, int mode, const BsrTask* tasks, uint32_t n_tasks, const BsrRun* runs,
                        const uint32_t* tile_cols, const void* bt0, const void* bt1, void* ws, bool narrow) {
    if (n_tasks == 0) return hipSuccess;
    const dim3 grid(n_tasks);
#define MQ_S_BSR(M_)                                                                                  \
    if (narrow)                                                                                       \
        hipLaunchKernelGGL((s_bsr_kernel<M_, true>), grid, dim3(BsrStep<M_>::NT), 0, st, tasks, runs, tile_cols, bt0, bt1, ws);  \
    else                                                                                              \
        hipLaunchKernelGGL((s_bsr_kernel<M_, false>), grid, dim3(BsrStep<M_>::NT), 0, st, tasks, runs, tile_cols, bt0, bt1, ws)
    switch (mode) {
        case MODE_F64:
            MQ_S_BSR(MODE_F64);
            break;
        case MODE_F32:
            MQ_S_BSR(MODE_F32);
            break;
        case MODE_BF16X3:
            MQ_S_BSR(MODE_BF16X3);
            break;
        default:
            return hipErrorInvalidValue;
    }
#undef MQ_S_BSR
    return hipGetLastError();
}

}  // namespace mq
