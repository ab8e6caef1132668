// Stacked T-stage GEMM of the grouped sigma and right boundary steps on gfx950 MFMA:
//
//   T_D[pair rows, keys] = psi blocks (stacked row units) * R cohort      one task per right cohort
//
// The tasks are the stacked 128 x 128 and 64 x 64 tasks of the generic grouped GEMM (GemmTask / GemmRow /
// GemmSeg, one segment, no A / B remaps, no beta): the psi blocks that meet one right cohort are
// the row units of the task, the cohort (or a Hermitian partner block, transposed and scaled) is B,
// and every 16-row block is stored to its own pair slab through the unit's column map.  This
// kernel is the lean form of that case (the generic kernel keeps every other task shape):
//
//   * operands are staged k-contiguous, A as [m][k] and B as [n][k] (16 keys + a 16-byte pad per
//     row), and each lane reads the 4 consecutive keys it needs for the 4 MFMA k-steps of a 16-key
//     step with one 16-byte LDS read: lane group lk takes keys 4 lk .. 4 lk + 3 and k-step t uses
//     key 4 lk + t, for A and B alike (the sum over k does not depend on the order);
//   * with 128 x 128 tiles thread t stages row t % 128 of A (8 keys: one row unit, one address
//     stream) and column t / 2 of B (8 keys: one contiguous 64-byte run of a non-transposed
//     cohort, four 16-byte loads); with 64 x 64 tiles row t % 64 and column t / 4, 4 keys each,
//     so the per-element address work of the generic kernel is gone;
//   * keys beyond the segment read the last key and are zeroed on the A side only; rows and
//     columns beyond the tile's range read clamped, finite data into outputs that are not stored.
//
// MODE_F64: FP64 operands in LDS, v_mfma_f64_16x16x4f64; MODE_F32: FP32 in LDS (converted while
// staged, A scaled by its unit and segment factors), v_mfma_f32_16x16x4f32; MODE_BF16X3: each FP32
// value split while staged into hi = bf16(x), lo = bf16(x - hi) (gfx950's v_cvt_pk_bf16_f32, round to
// nearest even) and three v_mfma_f32_16x16x16bf16 products per block and 16-key step (hi*lo + lo*hi +
// hi*hi, FP32 accumulation: the S stage's split-product scheme; lane group lk supplies keys
// 4 lk .. 4 lk + 3 as one 8-byte LDS read).  C is FP64 or FP32.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "kernels.hpp"

namespace mq {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef double d2_a8 __attribute__((ext_vector_type(2), aligned(8)));   // 8-byte aligned global runs
typedef short s4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));

constexpr int TK = 16, TT = GEMM_THREADS;

template <int MODE> struct TsTraits;
template <> struct TsTraits<MODE_F64> { typedef double T; typedef d4 Acc; static constexpr int P = TK + 2; };
template <> struct TsTraits<MODE_F32> { typedef float T; typedef f4 Acc; static constexpr int P = TK + 4; };

template <> struct TsTraits<MODE_BF16X3> { typedef float T; typedef f4 Acc; static constexpr int P = TK + 8; };

template <int MODE, int BM> struct TsSmem {
    typedef typename TsTraits<MODE>::T T;
    T a[BM][TsTraits<MODE>::P];
    T b[BM][TsTraits<MODE>::P];
};
// BF16X3: hi and lo bf16 of A and B, rows of 16 keys + 8 pad (48 bytes, 16-byte aligned runs)
template <int BM> struct TsSmem<MODE_BF16X3, BM> {
    static constexpr int P = TsTraits<MODE_BF16X3>::P;
    uint16_t ahi[BM][P], alo[BM][P], bhi[BM][P], blo[BM][P];
};

// waves per SIMD the kernel is compiled for (register budget): 128 x 128 tiles hold 16 blocks of
// accumulators per wave, 64 x 64 tiles 4
constexpr int ts_waves(int mode, int bm) {
    return bm == 64 ? 4 : mode == MODE_F32 ? 3 : mode == MODE_F64 ? 1 : 2;
}

// hi = bf16(x), lo = bf16(x - hi) of two elements, each pair packed lower element first
__device__ inline void split2(float x0, float x1, uint32_t& hi, uint32_t& lo) {
    hi = __builtin_bit_cast(uint32_t, bf2{(__bf16)x0, (__bf16)x1});
    lo = __builtin_bit_cast(uint32_t, bf2{(__bf16)(x0 - __uint_as_float(hi << 16)),
                                          (__bf16)(x1 - __uint_as_float(hi & 0xffff0000u))});
}

// The same of two elements of B, held in FP64, by one rule for both kernels: hi is the bf16 nearest to the
// FP32 value, in the first 16-key step nearest to the FP64 value; lo = bf16(FP32 value - hi).  The two differ
// where the FP32 value lies halfway between two bf16 and the FP64 value does not; hi + lo is the FP32 value
// to the same 17 bits either way.  The empty asm hides where the FP32 values come from: a conversion of them
// to bf16 would otherwise be made from the FP64 values wherever the compiler sees those.
template <bool FIRST>
__device__ inline void split_b(double d0, double d1, uint32_t& hi, uint32_t& lo) {
    float x0 = float(d0), x1 = float(d1);
    asm("" : "+v"(x0), "+v"(x1));
    hi = FIRST ? __builtin_bit_cast(uint32_t, bf2{(__bf16)d0, (__bf16)d1})
               : __builtin_bit_cast(uint32_t, bf2{(__bf16)x0, (__bf16)x1});
    lo = __builtin_bit_cast(uint32_t, bf2{(__bf16)(x0 - __uint_as_float(hi << 16)),
                                          (__bf16)(x1 - __uint_as_float(hi & 0xffff0000u))});
}

__device__ inline uint32_t task_of(const GemmTask* tasks, uint32_t n_tasks, const uint32_t* tile_task, uint32_t tile) {
    if (tile_task) return tile_task[tile];
    if (n_tasks == gridDim.x) return tile;
    uint32_t lo = 0, hi = n_tasks;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (tasks[mid].tile_begin <= tile) lo = mid; else hi = mid;
    }
    return lo;
}

// BM x BM tiles (BM = 128 or 64), 2 x 2 waves of WB x WB 16 x 16 blocks; each thread stages KPT
// keys of one A row and of one B column per 16-key step
template <int MODE, typename TC, int BM>
__global__ __launch_bounds__(TT) __attribute__((amdgpu_waves_per_eu(ts_waves(MODE, BM))))
void t_stack_kernel(const GemmTask* __restrict__ tasks, uint32_t n_tasks, const GemmSeg* __restrict__ segs,
                    Bases bases, GemmTables tables, const uint32_t* __restrict__ tile_task) {
    typedef typename TsTraits<MODE>::T T;
    typedef typename TsTraits<MODE>::Acc Acc;
    constexpr int TM = BM, TN = BM, KPT = BM / 16, WB = BM / 32, BT = TK / KPT;
    static_assert(BM == 128 || BM == 64, "tile");
    __shared__ __align__(16) TsSmem<MODE, BM> sm[2];
    const uint32_t* __restrict__ maps = tables.maps;
    const GemmRow* __restrict__ rows = tables.rows;

    const uint32_t tile = xcd_tile_cyclic<32>(blockIdx.x, gridDim.x);
    const GemmTask tk = tasks[task_of(tasks, n_tasks, tile_task, tile)];
    const GemmSeg sg = segs[tk.seg0];
    const uint32_t M = tk.M, N = tk.N, K = sg.K;
    const uint32_t local = tile - tk.tile_begin, tiles_m = (M + TM - 1) / TM;
    const uint32_t m0 = (local % tiles_m) * TM, n0 = (local / tiles_m) * TN;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave & 1) * (BM / 2), wn = (wave >> 1) * (BM / 2);
    const int l16 = lane & 15, lk = lane >> 4;

    // A: row a_m of the tile, KPT keys from a_k; its row unit's psi block row (clamped into the block)
    const int a_m = tid % TM, a_k = (tid / TM) * KPT;
    const double* __restrict__ A = bases.p[sg.a_base] + sg.a_off;
    const double* a_row;
    uint64_t a_sk;
    T a_sc;
    {
        const uint32_t m = min(m0 + uint32_t(a_m), M - 1);
        const GemmRow R = rows[maps[tk.rowunit + m / 16]];
        const uint32_t i = min(m - R.row0, R.nrows - 1);
        a_row = A + R.a_src + uint64_t(i) * R.a_si;
        a_sk = R.a_sk;
        a_sc = T(R.a_scale * sg.alpha);
    }
    // B: column b_n of the tile (clamped into op(B)), KPT keys from b_k
    const int b_n = tid / BT, b_k = (tid % BT) * KPT;
    const double* __restrict__ B = bases.p[sg.b_base] + sg.b_off;
    const uint32_t bn = min(n0 + uint32_t(b_n), N - 1);
    const bool tb = sg.trans_b;
    const double* b_col = tb ? B + bn : B + uint64_t(bn) * sg.ldb;   // op(B)(k, n) = b_col[k * (tb ? ldb : 1)]
    const uint64_t b_sk = tb ? sg.ldb : 1;

    Acc acc[WB][WB];
#pragma unroll
    for (int i = 0; i < WB; ++i)
#pragma unroll
        for (int j = 0; j < WB; ++j) acc[i][j] = Acc{0, 0, 0, 0};

    double va[KPT], vb[KPT];
    bool part = false;   // the staged step holds keys beyond K
    auto gload = [&](uint32_t k0) {
        part = k0 + TK > K;
        if (!part) {
            const double* pa = a_row + uint64_t(k0 + a_k) * a_sk;
#pragma unroll
            for (int e = 0; e < KPT; ++e) va[e] = pa[uint64_t(e) * a_sk];
            if (!tb) {
                const d2_a8* pb = reinterpret_cast<const d2_a8*>(b_col + k0 + b_k);
#pragma unroll
                for (int v = 0; v < KPT / 2; ++v) {
                    const d2_a8 x = pb[v];
                    vb[2 * v] = x[0];
                    vb[2 * v + 1] = x[1];
                }
            } else {
                const double* pb = b_col + uint64_t(k0 + b_k) * b_sk;
#pragma unroll
                for (int e = 0; e < KPT; ++e) vb[e] = pb[uint64_t(e) * b_sk];
            }
        } else {
#pragma unroll
            for (int e = 0; e < KPT; ++e) {
                va[e] = a_row[uint64_t(min(k0 + uint32_t(a_k + e), K - 1)) * a_sk];
                vb[e] = b_col[uint64_t(min(k0 + uint32_t(b_k + e), K - 1)) * b_sk];
            }
        }
    };
    auto lstore = [&](int buf, uint32_t k0, auto first) {
        TsSmem<MODE, BM>& s = sm[buf];
        T xa[KPT], xb[KPT];
#pragma unroll
        for (int e = 0; e < KPT; ++e) {
            xa[e] = T(va[e]) * a_sc;
            if (part && k0 + uint32_t(a_k + e) >= K) xa[e] = T(0);
            xb[e] = T(vb[e]);
        }
        if constexpr (MODE == MODE_BF16X3) {
            uint32_t ah[KPT / 2], al[KPT / 2], bh[KPT / 2], bl[KPT / 2];
#pragma unroll
            for (int e = 0; e < KPT / 2; ++e) {
                split2(xa[2 * e], xa[2 * e + 1], ah[e], al[e]);
                split_b<decltype(first)::value>(vb[2 * e], vb[2 * e + 1], bh[e], bl[e]);
            }
            if constexpr (KPT == 8) {
                *reinterpret_cast<uint4*>(&s.ahi[a_m][a_k]) = uint4{ah[0], ah[1], ah[2], ah[3]};
                *reinterpret_cast<uint4*>(&s.alo[a_m][a_k]) = uint4{al[0], al[1], al[2], al[3]};
                *reinterpret_cast<uint4*>(&s.bhi[b_n][b_k]) = uint4{bh[0], bh[1], bh[2], bh[3]};
                *reinterpret_cast<uint4*>(&s.blo[b_n][b_k]) = uint4{bl[0], bl[1], bl[2], bl[3]};
            } else {
                *reinterpret_cast<uint2*>(&s.ahi[a_m][a_k]) = uint2{ah[0], ah[1]};
                *reinterpret_cast<uint2*>(&s.alo[a_m][a_k]) = uint2{al[0], al[1]};
                *reinterpret_cast<uint2*>(&s.bhi[b_n][b_k]) = uint2{bh[0], bh[1]};
                *reinterpret_cast<uint2*>(&s.blo[b_n][b_k]) = uint2{bl[0], bl[1]};
            }
        } else if constexpr (MODE == MODE_F32) {
#pragma unroll
            for (int v = 0; v < KPT / 4; ++v) {
                *reinterpret_cast<float4*>(&s.a[a_m][a_k + 4 * v]) = float4{xa[4 * v], xa[4 * v + 1], xa[4 * v + 2], xa[4 * v + 3]};
                *reinterpret_cast<float4*>(&s.b[b_n][b_k + 4 * v]) = float4{xb[4 * v], xb[4 * v + 1], xb[4 * v + 2], xb[4 * v + 3]};
            }
        } else {
#pragma unroll
            for (int v = 0; v < KPT / 2; ++v) {
                *reinterpret_cast<double2*>(&s.a[a_m][a_k + 2 * v]) = double2{xa[2 * v], xa[2 * v + 1]};
                *reinterpret_cast<double2*>(&s.b[b_n][b_k + 2 * v]) = double2{xb[2 * v], xb[2 * v + 1]};
            }
        }
    };
    auto compute = [&](int buf) {
        const TsSmem<MODE, BM>& s = sm[buf];
        if constexpr (MODE == MODE_BF16X3) {
            s4 ah[WB], al[WB], bh[WB], bl[WB];   // keys 4 lk .. 4 lk + 3 of one row / column
#pragma unroll
            for (int i = 0; i < WB; ++i) {
                ah[i] = *reinterpret_cast<const s4*>(&s.ahi[wm + 16 * i + l16][4 * lk]);
                al[i] = *reinterpret_cast<const s4*>(&s.alo[wm + 16 * i + l16][4 * lk]);
                bh[i] = *reinterpret_cast<const s4*>(&s.bhi[wn + 16 * i + l16][4 * lk]);
                bl[i] = *reinterpret_cast<const s4*>(&s.blo[wn + 16 * i + l16][4 * lk]);
            }
#pragma unroll
            for (int i = 0; i < WB; ++i)
#pragma unroll
                for (int j = 0; j < WB; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah[i], bl[j], acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(al[i], bh[j], acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah[i], bh[j], acc[i][j], 0, 0, 0);
                }
        } else {
            T a[WB][4], b[WB][4];   // [block][k-step]: keys 4 lk + t
#pragma unroll
            for (int i = 0; i < WB; ++i) {
                const T* pa = &s.a[wm + 16 * i + l16][4 * lk];
                const T* pb = &s.b[wn + 16 * i + l16][4 * lk];
                if constexpr (MODE == MODE_F32) {
                    const float4 x = *reinterpret_cast<const float4*>(pa);
                    const float4 y = *reinterpret_cast<const float4*>(pb);
                    a[i][0] = x.x, a[i][1] = x.y, a[i][2] = x.z, a[i][3] = x.w;
                    b[i][0] = y.x, b[i][1] = y.y, b[i][2] = y.z, b[i][3] = y.w;
                } else {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const double2 x = *reinterpret_cast<const double2*>(pa + 2 * h);
                        const double2 y = *reinterpret_cast<const double2*>(pb + 2 * h);
                        a[i][2 * h] = x.x, a[i][2 * h + 1] = x.y;
                        b[i][2 * h] = y.x, b[i][2 * h + 1] = y.y;
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int i = 0; i < WB; ++i)
#pragma unroll
                    for (int j = 0; j < WB; ++j) {
                        if constexpr (MODE == MODE_F64)
                            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][t], b[j][t], acc[i][j], 0, 0, 0);
                        else
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][t], b[j][t], acc[i][j], 0, 0, 0);
                    }
        }
    };

    // ---- the K steps: compute step k0 while step k0 + 16 loads (one barrier per step)
    if (K > 0) {
        uint32_t k0 = 0;
        gload(k0);
        lstore(0, k0, std::true_type{});
        __syncthreads();
        int buf = 0;
        while (true) {
            const uint32_t k1 = k0 + TK;
            const bool more = k1 < K;
            if (more) gload(k1);
            compute(buf);
            if (!more) break;
            lstore(buf ^ 1, k1, std::false_type{});
            __syncthreads();
            buf ^= 1;
            k0 = k1;
        }
    }

    // ---- epilogue: each 16-row block of the wave lies in one row unit, stored to its slab through
    // the unit's column map; the 4 FP32 accumulator rows of a lane are consecutive (one 16-byte
    // store when all are inside the unit)
    TC* __restrict__ C = reinterpret_cast<TC*>(bases.p[tk.c_base]) + tk.c_off;
    // the lane's column of block j: its column block in the unit's column map and the column in it
    // (the same for every row block)
    uint32_t cblk[WB], cin[WB];
    {
        const uint32_t cbw = max(tk.cbw, 1u);
#pragma unroll
        for (int j = 0; j < WB; ++j) {
            const uint32_t gn = n0 + wn + 16 * j + l16;
            cblk[j] = gn / cbw;
            cin[j] = gn - cblk[j] * cbw;
        }
    }
#pragma unroll
    for (int i = 0; i < WB; ++i) {
        const uint32_t mb = m0 + wm + 16 * i;
        if (mb >= M) continue;
        const GemmRow R = rows[maps[tk.rowunit + mb / 16]];
#pragma unroll
        for (int j = 0; j < WB; ++j) {
            const uint32_t gn = n0 + wn + 16 * j + l16;
            if (gn >= N) continue;
            uint64_t coff;
            if (R.cmap != MAP_NONE) {
                coff = uint64_t(maps[R.cmap + cblk[j]]) * R.cldk + uint64_t(cin[j]) * R.ldc;
            } else {
                coff = uint64_t(gn) * R.ldc;
            }
            TC* __restrict__ Cc = C + R.c_src + coff;
            if constexpr (MODE != MODE_F64 && std::is_same<TC, float>::value) {
                const uint32_t li0 = mb + 4 * lk - R.row0;
                if (R.c_si == 1 && mb + 4 * lk + 3 < M && li0 + 3 < R.nrows) {
                    typedef float __attribute__((ext_vector_type(4), aligned(4))) f4_a4;
                    *reinterpret_cast<f4_a4*>(Cc + li0) = f4_a4{acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
                    continue;
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t gm = mb + (MODE == MODE_F64 ? 4 * r + lk : 4 * lk + r);
                const uint32_t li = gm - R.row0;
                if (gm < M && li < R.nrows) Cc[uint64_t(li) * R.c_si] = TC(acc[i][j][r]);
            }
        }
    }
}

// The streamed form of the stacked tasks: a workgroup of NW waves keeps 16 RB rows of A in LDS for the
// whole K range (K <= KP) and streams a strip of `strip` columns past them; each wave takes chunks of
// WC = 16 CB columns.  A step's B (WC columns x 16 keys) goes from memory to the wave's own part of LDS
// ([n][k], the next step's loads in flight meanwhile) and from there into the MFMA lane layout, so no
// barrier follows the staging of A and the waves drift freely: stores of one overlap products of
// another.
//
// What bounds it: the stores of T_D (in segments of one sector's rows), in FP64 the matrix cores
// beside them.  T's products are short (K is one sector: 75 keys by flops at SU2U1 L=24 m=1000) and its
// output large, so tiles of 128 x 128 spent most of their time filling and draining, in FP64 at one
// wave per SIMD.  Here A is read, scaled, converted and (BF16X3) split once per strip instead of once
// per column tile, and every B element is read and converted by one wave.  Neighbouring lanes always
// touch neighbouring addresses, which the vector cache's rate of one line per cycle asks for: B by
// runs of 16 keys, and T_D along its rows, with the MFMA operands exchanged (D = B^T A^T: lane l16 is
// a row of A, the four accumulators are columns).  T stage in ms, t_stack_kernel -> this: SU2U1 L=30
// m=1500 FP64 18.5 -> 10.1, BF16X3 5.5 -> 5.1; L=24 m=1000 4.4 -> 2.3 and 1.40 -> 1.30; L=16 m=256
// BF16X3 0.061 -> 0.051.  (B straight from memory in the MFMA layout, whose neighbouring lanes are
// different columns: FP64 11.0, BF16X3 5.9 at L=30; stores along the columns: slower still.)
//
// Classes by K: 64 rows of A up to K = 64 take 34 KB in FP64, three workgroups of 4 waves per CU;
// up to 144 75 KB, one workgroup of 8 waves; up to 288 32 rows fit beside the 8 waves' buffers.
//
// Same products, key slots and step order as t_stack_kernel: bitwise the same T_D.
// LDS accesses of one wave execute in program order; this keeps the compiler from moving them
__device__ inline void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
template <int MODE> constexpr int TP_PAD = MODE == MODE_F64 ? 2 : MODE == MODE_F32 ? 4 : 8;   // odd number of 16-byte runs per row

template <int MODE, typename TC, int KP, int RB, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(MODE == MODE_BF16X3 ? 4 : MODE == MODE_F64 && NW == 8 ? 2 : 3)))
void t_stream_kernel(const GemmTask* __restrict__ tasks, uint32_t n_tasks, const GemmSeg* __restrict__ segs,
                     Bases bases, GemmTables tables, const uint32_t* __restrict__ tile_task, uint32_t strip) {
    typedef typename TsTraits<MODE>::T T;
    typedef typename TsTraits<MODE>::Acc Acc;
    constexpr bool BF = MODE == MODE_BF16X3;
    constexpr int CB = 2, TM = 16 * RB, WC = 16 * CB, KPT = TK * TM / (64 * NW);
    constexpr int P = KP + TP_PAD<MODE>, PB = TK + TP_PAD<MODE>;
    static_assert(KPT >= 1 && KP % TK == 0, "A staging");
    typedef typename std::conditional<BF, uint16_t, T>::type E;
    __shared__ __align__(16) E sa[BF ? 2 : 1][TM][P];          // BF16X3: hi, lo
    struct Wave {   // one wave's own: a step of B, or (between chunks) the C offsets of a chunk's columns
        union {
            E b[BF ? 2 : 1][WC][PB];
            uint64_t off[RB][WC];
        };
    };
    __shared__ __align__(16) Wave sw[NW];
    const uint32_t* __restrict__ maps = tables.maps;
    const GemmRow* __restrict__ rows = tables.rows;

    const uint32_t tile = xcd_tile_cyclic<8>(blockIdx.x, gridDim.x);
    const GemmTask tk = tasks[task_of(tasks, n_tasks, tile_task, tile)];
    const GemmSeg sg = segs[tk.seg0];
    const uint32_t M = tk.M, N = tk.N, K = sg.K;
    const uint32_t local = tile - tk.tile_begin, tiles_m = (M + TM - 1) / TM;
    const uint32_t m0 = (local % tiles_m) * TM, n_begin = (local / tiles_m) * strip, n_end = min(N, n_begin + strip);

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, lk = lane >> 4;
    const uint32_t steps = (K + TK - 1) / TK;

    // ---- A: thread t stages row t % TM, keys (t / TM) KPT .. of every step (keys beyond K as zero)
    {
        const int am = tid % TM, ak = (tid / TM) * KPT;
        const uint32_t m = min(m0 + uint32_t(am), M - 1);
        const GemmRow R = rows[maps[tk.rowunit + m / 16]];
        const uint32_t i = min(m - R.row0, R.nrows - 1);
        const double* __restrict__ a_row = bases.p[sg.a_base] + sg.a_off + R.a_src + uint64_t(i) * R.a_si;
        const T a_sc = T(R.a_scale * sg.alpha);
#pragma unroll 2
        for (uint32_t s = 0; s < steps; ++s) {
            T x[KPT];
#pragma unroll
            for (int e = 0; e < KPT; ++e) {
                const uint32_t k = s * TK + ak + e;
                x[e] = T(a_row[uint64_t(min(k, K - 1)) * R.a_sk]) * a_sc;
                if (k >= K) x[e] = T(0);
            }
            E* d = &sa[0][am][s * TK + ak];
#pragma unroll
            for (int e = 0; e < KPT; ++e) {
                if constexpr (BF) {
                    uint32_t h, l;
                    split2(x[e], 0.f, h, l);
                    d[e] = uint16_t(h);
                    d[TM * P + e] = uint16_t(l);
                } else {
                    d[e] = x[e];
                }
            }
        }
    }
    __syncthreads();

    const double* __restrict__ B = bases.p[sg.b_base] + sg.b_off;
    TC* __restrict__ C = reinterpret_cast<TC*>(bases.p[tk.c_base]) + tk.c_off;
    const uint32_t cbw = max(tk.cbw, 1u);
    E(*wb)[WC][PB] = sw[wave].b;

    // ---- where T_D's elements go.  The lane's row of every 16-row block: its offset in the block's unit,
    // ~0 if it is padding.
    uint32_t rowoff[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        const uint32_t mb = min(m0 + 16 * i, M - 16);
        const GemmRow& R = rows[maps[tk.rowunit + mb / 16]];
        const uint32_t li = mb + l16 - R.row0;
        rowoff[i] = m0 + 16 * i < M && li < R.nrows ? li * R.c_si : ~0u;
    }
    // The units whose column offsets the lane computes: column lane % 32 of a chunk, row blocks
    // lane / 32 + 2 p (a chunk's offsets go through LDS; their map entries are loaded at its start)
    static_assert(WC == 32 && RB % 2 == 0, "two row blocks per pass");
    constexpr int NP = RB / 2;
    uint64_t u_src[NP];
    uint32_t u_cmap[NP], u_cldk[NP], u_ldc[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const GemmRow& R = rows[maps[tk.rowunit + min(m0 + 16 * (lane / 32 + 2 * p), M - 16) / 16]];
        u_src[p] = R.c_src;
        u_cmap[p] = R.cmap;
        u_cldk[p] = R.cldk;
        u_ldc[p] = R.ldc;
    }

    auto body = [&](auto trans) {
        constexpr bool TB = decltype(trans)::value;
        const uint64_t ldb = sg.ldb;
        // B of a step, NV pairs of doubles per lane: stored cohort (k contiguous): pair v is keys
        // 2 (lane % 8) of column lane / 8 + 8 v; transposed (n contiguous): columns 2 (lane % (WC / 2)),
        // key lane / (WC / 2) + (128 / WC) v
        constexpr int NV = WC / 8;
        d2_a8 vb[NV];
        const int b_n = TB ? 2 * (lane % (WC / 2)) : lane / 8, b_k = TB ? lane / (WC / 2) : 2 * (lane % 8);
        auto load = [&](uint32_t c, uint32_t s) {   // keys beyond K and columns beyond N read the last one
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                if constexpr (TB) {
                    const uint32_t n = c + b_n;
                    const double* p = B + uint64_t(min(s * TK + b_k + (128 / WC) * v, K - 1)) * ldb;
                    vb[v][0] = p[min(n, N - 1)];
                    vb[v][1] = p[min(n + 1, N - 1)];
                } else {
                    const double* p = B + uint64_t(min(c + b_n + 8 * v, N - 1)) * ldb;
                    const uint32_t k = s * TK + b_k;
                    if ((s + 1) * TK <= K) {
                        vb[v] = *reinterpret_cast<const d2_a8*>(p + k);
                    } else {
                        vb[v][0] = p[min(k, K - 1)];
                        vb[v][1] = p[min(k + 1, K - 1)];
                    }
                }
            }
        };
        // BF16X3: the first step's split differs only where an FP32 value lies halfway between two bf16, so its
        // longer conversion runs only for a first step that holds one (one in a hundred)
        auto put = [&](auto first) {   // the loaded step into the wave's LDS, in the arithmetic's type
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const T x = T(vb[v][0]), y = T(vb[v][1]);
                if constexpr (TB) {
                    const int k = b_k + (128 / WC) * v;
                    if constexpr (BF) {
                        uint32_t h, l;
                        split_b<decltype(first)::value>(vb[v][0], vb[v][1], h, l);
                        wb[0][b_n][k] = uint16_t(h);
                        wb[0][b_n + 1][k] = uint16_t(h >> 16);
                        wb[1][b_n][k] = uint16_t(l);
                        wb[1][b_n + 1][k] = uint16_t(l >> 16);
                    } else {
                        wb[0][b_n][k] = x;
                        wb[0][b_n + 1][k] = y;
                    }
                } else {
                    const int n = b_n + 8 * v;
                    if constexpr (BF) {
                        uint32_t h, l;
                        split_b<decltype(first)::value>(vb[v][0], vb[v][1], h, l);
                        *reinterpret_cast<uint32_t*>(&wb[0][n][b_k]) = h;
                        *reinterpret_cast<uint32_t*>(&wb[1][n][b_k]) = l;
                    } else {
                        typedef T t2 __attribute__((ext_vector_type(2)));
                        *reinterpret_cast<t2*>(&wb[0][n][b_k]) = t2{x, y};
                    }
                }
            }
        };
        uint32_t c = n_begin + wave * WC;
        if (c >= n_end) return;
        load(c, 0);
        while (true) {
            Acc acc[RB][CB];
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int j = 0; j < CB; ++j) acc[i][j] = Acc{0, 0, 0, 0};
            const uint32_t oc = min(c + lane % 32, n_end - 1), oblk = oc / cbw, oin = oc - oblk * cbw;
            uint32_t om[NP];
#pragma unroll
            for (int p = 0; p < NP; ++p) om[p] = u_cmap[p] != MAP_NONE ? maps[u_cmap[p] + oblk] : 0u;
            const uint32_t next = c + NW * WC;
            for (uint32_t s = 0; s < steps; ++s) {
                bool halfway = false;
                if (BF && s == 0) {
#pragma unroll
                    for (int v = 0; v < NV; ++v)
#pragma unroll
                        for (int e = 0; e < 2; ++e)
                            halfway = halfway || (__float_as_uint(float(vb[v][e])) & 0xffffu) == 0x8000u;
                    halfway = __any(halfway);
                }
                if (halfway) put(std::true_type{});
                else put(std::false_type{});
                // the next step's loads (or the next chunk's first; past the strip the last again)
                const bool last = s + 1 == steps;
                load(last ? min(next, n_end - 1) : c, last ? 0 : s + 1);
                wave_fence();   // the wave's LDS accesses stay in this order
                if constexpr (BF) {
                    s4 bh[CB], bl[CB];
#pragma unroll
                    for (int j = 0; j < CB; ++j) {
                        bh[j] = *reinterpret_cast<const s4*>(&wb[0][16 * j + l16][4 * lk]);
                        bl[j] = *reinterpret_cast<const s4*>(&wb[1][16 * j + l16][4 * lk]);
                    }
#pragma unroll
                    for (int i = 0; i < RB; ++i) {
                        const s4 ah = *reinterpret_cast<const s4*>(&sa[0][16 * i + l16][s * TK + 4 * lk]);
                        const s4 al = *reinterpret_cast<const s4*>(&sa[1][16 * i + l16][s * TK + 4 * lk]);
#pragma unroll
                        for (int j = 0; j < CB; ++j) {
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bl[j], ah, acc[i][j], 0, 0, 0);
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bh[j], al, acc[i][j], 0, 0, 0);
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(bh[j], ah, acc[i][j], 0, 0, 0);
                        }
                    }
                } else {
                    typedef T tv __attribute__((ext_vector_type(16 / sizeof(T))));
                    constexpr int VN = 16 / sizeof(T);
                    T a[RB][4], bb[CB][4];
#pragma unroll
                    for (int h = 0; h < 4 / VN; ++h) {
#pragma unroll
                        for (int j = 0; j < CB; ++j) {
                            const tv x = *reinterpret_cast<const tv*>(&wb[0][16 * j + l16][4 * lk + VN * h]);
#pragma unroll
                            for (int e = 0; e < VN; ++e) bb[j][VN * h + e] = x[e];
                        }
#pragma unroll
                        for (int i = 0; i < RB; ++i) {
                            const tv x = *reinterpret_cast<const tv*>(&sa[0][16 * i + l16][s * TK + 4 * lk + VN * h]);
#pragma unroll
                            for (int e = 0; e < VN; ++e) a[i][VN * h + e] = x[e];
                        }
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int i = 0; i < RB; ++i)
#pragma unroll
                            for (int j = 0; j < CB; ++j) {
                                if constexpr (MODE == MODE_F64)
                                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bb[j][e], a[i][e], acc[i][j], 0, 0, 0);
                                else
                                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bb[j][e], a[i][e], acc[i][j], 0, 0, 0);
                            }
                }
                wave_fence();
            }
            // ---- store the chunk
#pragma unroll
            for (int p = 0; p < NP; ++p)
                sw[wave].off[lane / 32 + 2 * p][lane % 32] =
                    u_src[p] + (u_cmap[p] != MAP_NONE ? uint64_t(om[p]) * u_cldk[p] + uint64_t(oin) * u_ldc[p]
                                                      : uint64_t(oc) * u_ldc[p]);
            wave_fence();
            // D = B^T A^T: lane l16 is row l16 of every 16-row block, accumulator r of block j the column
            // 16 j + 4 r + lk (FP64) or 16 j + 4 lk + r
#pragma unroll
            for (int j = 0; j < CB; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int n = 16 * j + (MODE == MODE_F64 ? 4 * r + lk : 4 * lk + r);
                    if (c + n >= n_end) continue;
#pragma unroll
                    for (int i = 0; i < RB; ++i)
                        if (rowoff[i] != ~0u) C[sw[wave].off[i][n] + rowoff[i]] = TC(acc[i][j][r]);
                }
            wave_fence();
            c = next;
            if (c >= n_end) break;
        }
    };
    if (sg.trans_b) body(std::true_type{});
    else body(std::false_type{});
}

template <int MODE, typename TC>
hipError_t launch_t_stream_mode(hipStream_t st, int cls, const GemmTask* tasks, uint32_t n_tasks, const GemmSeg* segs,
                                uint32_t n_tiles, uint32_t strip, Bases bases, GemmTables tb,
                                const uint32_t* tile_task) {
#define MQ_T_STREAM(KP_, RB_, NW_)                                                                              \
    hipLaunchKernelGGL((t_stream_kernel<MODE, TC, KP_, RB_, NW_>), dim3(n_tiles), dim3(64 * NW_), 0, st, tasks, \
                       n_tasks, segs, bases, tb, tile_task, strip)
    switch (cls) {
        case 0: MQ_T_STREAM(T_STREAM_KMAX[0], T_STREAM_ROWS[0] / 16, 4); break;
        case 1: MQ_T_STREAM(T_STREAM_KMAX[1], T_STREAM_ROWS[1] / 16, 8); break;
        case 2: MQ_T_STREAM(T_STREAM_KMAX[2], T_STREAM_ROWS[2] / 16, 8); break;
        default: return hipErrorInvalidValue;
    }
#undef MQ_T_STREAM
    return hipGetLastError();
}

// The final stage of the boundary steps (FP64): one stacked task per new cohort, its blocks the row
// units, K segments over the physical states, each reading every unit's S_D slab through its block map
// (GemmSeg::amap):
//
//   right step  A(m, k) = S[.. + i + k lda] (rows contiguous), B(k, n) = bra[.. + n + k ldb]
//   left step   A(m, k) = S[.. + i lda + k] (keys contiguous), B(k, n) = bra[.. + k + n ldb]
//
// What bounds it: the bra side N is one sector, so a task is a tall product that reads S_D about once; the
// generic kernel spent its time on per-element addresses and on loads whose neighbouring lanes are
// different columns, one step ahead.  Here a thread stages 4 keys of one row of A and of one column of
// B, dealt so that neighbouring lanes read neighbouring addresses in either orientation, two steps
// ahead; 4 waves of 16 x 64 skip the column blocks beyond N alike.  SU2U1 L=30 m=1500 right step, final
// stage: 10.0 -> 3.6 ms; L=24 m=1000 left step: 2.8 -> 1.1 ms.
constexpr int RS_BM = 64, RS_BN = 64, RS_P = TK + 2;
__global__ __launch_bounds__(TT) __attribute__((amdgpu_waves_per_eu(3)))
void step_final_kernel(const GemmTask* __restrict__ tasks, uint32_t n_tasks, const GemmSeg* __restrict__ segs,
                       Bases bases, GemmTables tables, const uint32_t* __restrict__ tile_task) {
    __shared__ __align__(16) double sa[2][RS_BM][RS_P], sb[2][RS_BN][RS_P];
    const uint32_t* __restrict__ maps = tables.maps;
    const GemmRow* __restrict__ rows = tables.rows;

    const uint32_t tile = xcd_tile_cyclic<16>(blockIdx.x, gridDim.x);
    const GemmTask tk = tasks[task_of(tasks, n_tasks, tile_task, tile)];
    const uint32_t M = tk.M, N = tk.N;
    const uint32_t local = tile - tk.tile_begin;   // column tile fastest: a row panel's tiles share its S_D
    const uint32_t m0 = (local / tk.tiles_n) * RS_BM, n0 = (local % tk.tiles_n) * RS_BN;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, lk = lane >> 4;

    // the orientation is one for all segments of a task
    const bool ta = segs[tk.seg0].trans_a != 0, tb = segs[tk.seg0].trans_b != 0;
    const int a_m = ta ? tid >> 2 : tid & 63, a_k = 4 * (ta ? tid & 3 : tid >> 6);
    const int b_n = tb ? tid & 63 : tid >> 2, b_k = 4 * (tb ? tid >> 6 : tid & 3);
    uint32_t a_i, a_j;
    double a_rs;
    {
        const uint32_t m = min(m0 + uint32_t(a_m), M - 1);
        const GemmRow& R = rows[maps[tk.rowunit + m / 16]];
        a_i = min(m - R.row0, R.nrows - 1);
        a_j = R.jblk;
        a_rs = R.a_scale;
    }
    const uint32_t bn = min(n0 + uint32_t(b_n), N - 1);
    const int nj = int(min((N - n0 + 15) / 16, uint32_t(RS_BN / 16)));   // column blocks inside N (uniform)

    // cursor over the steps of all segments; a segment's row and column addresses
    uint32_t sgi = tk.seg0, k0 = 0;
    GemmSeg sg = segs[sgi];
    const double *a_row = nullptr, *b_col = nullptr;
    auto begin_seg = [&]() {
        a_row = bases.p[sg.a_base] + sg.a_off + uint64_t(maps[sg.amap + a_j]) * sg.bldk + uint64_t(a_i) * (ta ? sg.lda : 1u);
        b_col = bases.p[sg.b_base] + sg.b_off + uint64_t(bn) * (tb ? 1u : sg.ldb);
    };
    auto advance = [&]() {   // to the next step; false (and stays) at the last
        if (k0 + TK < sg.K) {
            k0 += TK;
            return true;
        }
        if (sgi + 1 >= tk.seg1) return false;
        sg = segs[++sgi];
        k0 = 0;
        begin_seg();
        return true;
    };
    struct Stage {
        double a[4], b[4];
        double sc;
        uint32_t k0, K;
    };
    auto load = [&](Stage& s) {   // keys beyond the segment read its last one
        s.k0 = k0;
        s.K = sg.K;
        s.sc = a_rs * sg.alpha;
        const uint64_t ask = ta ? 1u : sg.lda, bsk = tb ? sg.ldb : 1u;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            s.a[e] = a_row[uint64_t(min(k0 + uint32_t(a_k + e), sg.K - 1)) * ask];
            s.b[e] = b_col[uint64_t(min(k0 + uint32_t(b_k + e), sg.K - 1)) * bsk];
        }
    };
    auto store = [&](const Stage& s, int buf) {
        double x[4], y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = s.a[e] * s.sc, y[e] = s.b[e];
        if (s.k0 + TK > s.K) {   // keys beyond the segment: both zero (0 times an infinity of its last key is a NaN)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (s.k0 + a_k + e >= s.K) x[e] = 0.0;
                if (s.k0 + b_k + e >= s.K) y[e] = 0.0;
            }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            *reinterpret_cast<double2*>(&sa[buf][a_m][a_k + 2 * h]) = double2{x[2 * h], x[2 * h + 1]};
            *reinterpret_cast<double2*>(&sb[buf][b_n][b_k + 2 * h]) = double2{y[2 * h], y[2 * h + 1]};
        }
    };
    d4 acc[RS_BN / 16];
#pragma unroll
    for (int j = 0; j < RS_BN / 16; ++j) acc[j] = d4{0, 0, 0, 0};
    auto compute = [&](int buf) {
        double a[4];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const double2 x = *reinterpret_cast<const double2*>(&sa[buf][16 * wave + l16][4 * lk + 2 * h]);
            a[2 * h] = x.x, a[2 * h + 1] = x.y;
        }
#pragma unroll
        for (int j = 0; j < RS_BN / 16; ++j) {
            if (j >= nj) break;
            double b[4];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const double2 x = *reinterpret_cast<const double2*>(&sb[buf][16 * j + l16][4 * lk + 2 * h]);
                b[2 * h] = x.x, b[2 * h + 1] = x.y;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[e], b[e], acc[j], 0, 0, 0);
        }
    };
    // compute step t from one buffer, step t + 1 in registers, step t + 2's loads issued (past the last
    // step the loads repeat it, unused)
    begin_seg();
    Stage ga, gb;
    load(ga);
    bool has = advance();
    load(gb);
    store(ga, 0);
    __syncthreads();
    while (true) {
        const bool next = has && advance();
        load(ga);
        compute(0);
        if (!has) break;
        store(gb, 1);
        __syncthreads();
        has = next && advance();
        load(gb);
        compute(1);
        if (!next) break;
        store(ga, 0);
        __syncthreads();
    }

    // ---- the wave's 16 rows lie in one unit
    const uint32_t mb = m0 + 16 * wave;
    if (mb >= M) return;
    const GemmRow R = rows[maps[tk.rowunit + mb / 16]];
    double* __restrict__ C = bases.p[tk.c_base] + tk.c_off + R.c_src;
#pragma unroll
    for (int j = 0; j < RS_BN / 16; ++j) {
        const uint32_t gn = n0 + 16 * j + l16;
        if (gn >= N) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t li = mb + 4 * r + lk - R.row0;
            if (li < R.nrows) C[uint64_t(gn) * R.ldc + uint64_t(li) * R.c_si] = acc[j][r];
        }
    }
}

template <int BM>
hipError_t launch_t_tile(hipStream_t st, int mode, bool c_float, const GemmTask* tasks, uint32_t n_tasks,
                         const GemmSeg* segs, uint32_t n_tiles, Bases bases, GemmTables tb, const uint32_t* tile_task) {
    const dim3 grid(n_tiles), block(TT);
    if (mode == MODE_F64 && !c_float)
        hipLaunchKernelGGL((t_stack_kernel<MODE_F64, double, BM>), grid, block, 0, st, tasks, n_tasks, segs, bases, tb, tile_task);
    else if (mode == MODE_F32 && c_float)
        hipLaunchKernelGGL((t_stack_kernel<MODE_F32, float, BM>), grid, block, 0, st, tasks, n_tasks, segs, bases, tb, tile_task);
    else if (mode == MODE_BF16X3 && c_float)
        hipLaunchKernelGGL((t_stack_kernel<MODE_BF16X3, float, BM>), grid, block, 0, st, tasks, n_tasks, segs, bases, tb, tile_task);
    else if (mode == MODE_F32)
        hipLaunchKernelGGL((t_stack_kernel<MODE_F32, double, BM>), grid, block, 0, st, tasks, n_tasks, segs, bases, tb, tile_task);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace

hipError_t launch_step_final(hipStream_t st, const GemmTask* tasks, uint32_t n_tasks, const GemmSeg* segs, uint32_t n_tiles,
                             Bases bases, GemmTables tb, const uint32_t* tile_task) {
    if (n_tiles == 0) return hipSuccess;
    hipLaunchKernelGGL(step_final_kernel, dim3(n_tiles), dim3(TT), 0, st, tasks, n_tasks, segs, bases, tb, tile_task);
    return hipGetLastError();
}

hipError_t launch_t_stream(hipStream_t st, int cls, int mode, bool c_float, const GemmTask* tasks, uint32_t n_tasks,
                           const GemmSeg* segs, uint32_t n_tiles, uint32_t strip, Bases bases, GemmTables tb,
                           const uint32_t* tile_task) {
    if (n_tiles == 0) return hipSuccess;
    if (mode == MODE_F64 && !c_float)
        return launch_t_stream_mode<MODE_F64, double>(st, cls, tasks, n_tasks, segs, n_tiles, strip, bases, tb, tile_task);
    if (mode == MODE_F32 && c_float)
        return launch_t_stream_mode<MODE_F32, float>(st, cls, tasks, n_tasks, segs, n_tiles, strip, bases, tb, tile_task);
    if (mode == MODE_BF16X3 && c_float)
        return launch_t_stream_mode<MODE_BF16X3, float>(st, cls, tasks, n_tasks, segs, n_tiles, strip, bases, tb, tile_task);
    return hipErrorInvalidValue;
}

hipError_t launch_t_stack(hipStream_t st, int cfg, int mode, bool c_float, const GemmTask* tasks, uint32_t n_tasks,
                          const GemmSeg* segs, uint32_t n_tiles, Bases bases, GemmTables tb, const uint32_t* tile_task) {
    if (n_tiles == 0) return hipSuccess;
    if (cfg == GEMM_CFG_128x128)
        return launch_t_tile<128>(st, mode, c_float, tasks, n_tasks, segs, n_tiles, bases, tb, tile_task);
    if (cfg == GEMM_CFG_64x64)
        return launch_t_tile<64>(st, mode, c_float, tasks, n_tasks, segs, n_tiles, bases, tb, tile_task);
    return hipErrorInvalidValue;
}

}  // namespace mq
