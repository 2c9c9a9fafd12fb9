// gemm_f64.hip -- MatMul::matmul on Tensor<f64, ...> (stdlib/linalg/matrix.cleave:27-61
// with T = f64; Float covers f64, stdlib/num/num.cleave:50-51), single and
// batched, in all four trans_a / trans_b layouts, on the f64 matrix cores.
//
// v_mfma_f64_16x16x4f64: a wave multiplies a 16 x 4 block of A by a 4 x 16
// block of B into a 16 x 16 f64 accumulator, each lane supplying one double
// of each operand (A[l % 16][l / 16], B[l / 16][l % 16]) and holding four
// results, rows l / 16 + 4 v (v = 0..3) of column l % 16 (measured on
// gfx950: unlike the f32 16x16x4 form, whose lane holds four consecutive
// rows, the f64 form interleaves them).  On MI355X one such
// instruction keeps a SIMD's matrix core busy 64 cycles (FP64 matrix peak
// 78.6 TFLOP/s = 128 FLOP per CU-clock).
//
// With so much time per operand pair there is no LDS staging: a wave computes
// a (16 FM) x (16 FN) tile of C from register fragments that it loads from the
// caches, STEP of K at a time (FM FN x 16 STEP cycles of MFMA a step), PF steps
// ahead, and the other waves of its SIMD cover the rest of the loads' latency.
// The register-staged LDS tiles of 128 x 128 that this replaced were slower but
// for A.B^T with K of 16 to 128 (43 of 4031 x 267 x 64 194 against 212 us, 4096^2 x
// 64 53.5 against 53): 4096^3 A.B 2206 -> 1906 us, A.B^T 2428 -> 2235, 4095^3 A.B^T (rows
// not 16-byte aligned) 3412 -> 2230, and with few tiles 1000^3 167 -> 40, 256^3
// 45 -> 5, 64^2 x 10000 1586 -> 10, 8192 x 10 x 4096 660 -> 45.  The same LDS
// scheme on 64 x 64 tiles took 69-73 us at 1000^3.
//
// WK = 4: the workgroup's four waves take quarters of K, added in LDS in wave
// order.  WK = 1: they take a 2 x 2 block of tiles, sharing their fragments'
// lines in L1.  Past that K is cut into `slices` workgroups per tile; each
// publishes its partial tile and the last to arrive adds them in slice order
// (last_block.hpp).  The order of every sum depends on the shape alone.
//
// k order: over an 8-deep block, lane group h = lane / 16 takes k = 2h + s at
// MFMA s for A and B alike, so a k-contiguous operand is one 16-byte load per
// lane, fragment and block (V2; two 8-byte loads where its rows or base are
// not 16-byte aligned).  Of an m/n-contiguous operand lane i = lane % 16 loads
// the neighbouring rows FM i .. FM i + FM - 1 at once, one for each fragment,
// at any alignment; a group that would pass the last row starts that many rows
// before the end and computes rows that its neighbour has too, in the same
// order, and stores the same values.  Rows of a k-contiguous operand past the
// product are read from its last row and feed only entries that are not
// stored; k past K enters as zero on both sides.  Any M, N, K takes the same path (K = 0
// included: C = 0, the zero-filled accumulator of matrix.cleave:59).
#include <algorithm>

#include "common.hpp"
#include "gemm_common.hpp"
#include "last_block.hpp"

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));

constexpr int kThreads = 256;
constexpr int kCounters = 4096;  // tiles that may be cut along K
static __device__ uint32_t g_counters[kCounters];  // 0 between launches

// One operand of a wave: F fragments of 16 rows (of A, or columns of B) by 16
// doubles of K.  KC: k-contiguous in memory.
template <int F>
struct Group {
    typedef double type __attribute__((ext_vector_type(F), aligned(8)));
};
template <>
struct Group<1> {
    typedef double type;
};
template <int F, bool KC, bool V2, int STEP>
struct Frags {
    static constexpr int E = STEP / 4;  // doubles a lane holds of a fragment
    const double* p[KC ? F : 1];
    int64_t ld;
    int first, rows;

    // r0: the wave's first row; rows: the operand's.
    __device__ __forceinline__ void init(const double* base, int64_t pitch, int r0, int nrows, int lane) {
        ld = pitch;
        first = r0;
        rows = nrows;
        const int h = lane >> 4, i = lane & 15;
        if constexpr (KC) {
#pragma unroll
            for (int f = 0; f < F; ++f) p[f] = base + (int64_t)min(r0 + 16 * f + i, nrows - 1) * pitch + 2 * h;
        } else {
            p[0] = base + (int64_t)(2 * h) * pitch + min(r0 + F * i, nrows - F);
        }
    }
    // The operand's row that fragment f holds at index i.
    __device__ __forceinline__ int row(int f, int i) const {
        return KC ? first + 16 * f + i : min(first + F * i, rows - F) + f;
    }
    // v[f][2 b + s]: k = 8 b + 2 h + s of the step.
    __device__ __forceinline__ void load(int64_t k, double (&v)[F][E]) const {
        if constexpr (KC) {
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const double* q = p[f] + k;
#pragma unroll
                for (int b = 0; b < E / 2; ++b) {
                    if constexpr (V2) {
                        const d2 x = *reinterpret_cast<const d2*>(q + 8 * b);
                        v[f][2 * b] = x[0];
                        v[f][2 * b + 1] = x[1];
                    } else {
                        v[f][2 * b] = q[8 * b];
                        v[f][2 * b + 1] = q[8 * b + 1];
                    }
                }
            }
        } else {
#pragma unroll
            for (int e = 0; e < E; ++e) take(p[0] + (k + 8 * (e >> 1) + (e & 1)) * ld, e, v);
        }
    }
    // The step at k of a range that ends at k1 < k + STEP.
    __device__ __forceinline__ void load_tail(int64_t k, int64_t k1, int lane, double (&v)[F][E]) const {
        const int h = lane >> 4;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int64_t at = 8 * (e >> 1) + (e & 1);
            const bool in = k + at + 2 * h < k1;
            if constexpr (KC) {
#pragma unroll
                for (int f = 0; f < F; ++f) v[f][e] = in ? p[f][k + at] : 0.0;
            } else if (in) {
                take(p[0] + (k + at) * ld, e, v);
            } else {
#pragma unroll
                for (int f = 0; f < F; ++f) v[f][e] = 0.0;
            }
        }
    }
    __device__ __forceinline__ static void take(const double* q, int e, double (&v)[F][E]) {
        if constexpr (F == 1) {
            v[0][e] = *q;
        } else {
            const typename Group<F>::type x = *reinterpret_cast<const typename Group<F>::type*>(q);
#pragma unroll
            for (int f = 0; f < F; ++f) v[f][e] = x[f];
        }
    }
};

// `part`: tiles x slices partial tiles, unused with slices == 1.  A 1-D grid of
// tiles_m * tiles_n * batch * slices workgroups.
// (Two waves a SIMD for two k-contiguous operands on 4 x 4 fragments, which the
// compiler gives 268 registers otherwise.)
template <bool KCA, bool KCB, bool V2A, bool V2B, int FM, int FN, int WK, int PF, int STEP>
__global__ __launch_bounds__(kThreads, KCA && KCB && FM * FN == 16 && PF < 3 ? 2 : 1) void gemm_f64_kernel(
    const double* __restrict__ A, const double* __restrict__ B, double* __restrict__ C, int M, int N, int K,
    int64_t lda, int64_t ldb, int64_t sa, int64_t sb, int64_t sc, int tiles_m, int tiles_n, int batch, int slices,
    int64_t kslice, double* part) {
    static_assert(WK == 1 || WK == 4, "waves along K");
    constexpr int NF = FM * FN;
    __shared__ double red[WK > 1 ? (WK - 1) * NF * 4 * 64 : 1];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int b, tm, tn;  // b: batch entry and slice
    ch::block_coords(blockIdx.x, tiles_m, tiles_n, batch * slices, b, tm, tn);
    const int entry = b / slices, z = b - entry * slices;
    A += (int64_t)entry * sa;
    B += (int64_t)entry * sb;
    C += (int64_t)entry * sc;
    const int m0 = WK == 1 ? (tm * 2 + (wave >> 1)) * 16 * FM : tm * 16 * FM;
    const int n0 = WK == 1 ? (tn * 2 + (wave & 1)) * 16 * FN : tn * 16 * FN;

    int64_t k0 = z * kslice, k1 = min((int64_t)K, k0 + kslice);
    if constexpr (WK > 1) {
        const int64_t steps = (k1 - k0 + STEP - 1) / STEP, each = (steps + WK - 1) / WK * STEP;
        k0 += wave * each;
        k1 = min(k1, k0 + each);
    }

    d4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
    auto mfma = [&](const double (&a)[FM][STEP / 4], const double (&bb)[FN][STEP / 4]) {
#pragma unroll
        for (int t = 0; t < STEP / 4; ++t)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][t], bb[j][t], acc[i][j], 0, 0, 0);
    };

    Frags<FM, KCA, V2A, STEP> fa;
    Frags<FN, KCB, V2B, STEP> fb;
    fa.init(A, lda, m0, M, lane);
    fb.init(B, ldb, n0, N, lane);
    if (k0 < k1) {
        const int whole = (int)((k1 - k0) / STEP);
        double a[PF][FM][STEP / 4], bb[PF][FN][STEP / 4];
#pragma unroll
        for (int u = 0; u < PF; ++u)
            if (u < whole) {
                fa.load(k0 + u * STEP, a[u]);
                fb.load(k0 + u * STEP, bb[u]);
            }
        for (int t = 0; t < whole; t += PF) {
#pragma unroll
            for (int u = 0; u < PF; ++u)
                if (t + u < whole) {
                    mfma(a[u], bb[u]);
                    if (t + u + PF < whole) {
                        fa.load(k0 + (int64_t)(t + u + PF) * STEP, a[u]);
                        fb.load(k0 + (int64_t)(t + u + PF) * STEP, bb[u]);
                    }
                }
        }
        k0 += (int64_t)whole * STEP;
        if (k0 < k1) {
            fa.load_tail(k0, k1, lane, a[0]);
            fb.load_tail(k0, k1, lane, bb[0]);
            mfma(a[0], bb[0]);
        }
    }

    if constexpr (WK > 1) {
        if (wave > 0) {
#pragma unroll
            for (int f = 0; f < NF; ++f)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    red[(((wave - 1) * NF + f) * 4 + v) * 64 + lane] = acc[f / FN][f % FN][v];
        }
        __syncthreads();
        if (wave == 0) {
#pragma unroll
            for (int w = 0; w < WK - 1; ++w)
#pragma unroll
                for (int f = 0; f < NF; ++f)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        acc[f / FN][f % FN][v] += red[((w * NF + f) * 4 + v) * 64 + lane];
        }
    }

    // acc[i][j][v]: index lane / 16 + 4 v of A's fragment i, lane % 16 of B's fragment j.
    auto put = [&](int f, int v, double x) {
        const int m = fa.row(f / FN, (lane >> 4) + 4 * v), n = fb.row(f % FN, lane & 15);
        if ((!KCA || m < M) && (!KCB || n < N)) C[(int64_t)m * N + n] = x;
    };
    if (slices == 1) {
        if (WK > 1 && wave != 0) return;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if constexpr (KCB) {
#pragma unroll
                    for (int j = 0; j < FN; ++j) put(i * FN + j, v, acc[i][j][v]);
                } else {  // a lane holds FN neighbouring columns
                    const int m = fa.row(i, (lane >> 4) + 4 * v);
                    if (KCA && m >= M) continue;
                    typename Group<FN>::type q;
                    if constexpr (FN == 1) {
                        q = acc[i][0][v];
                    } else {
#pragma unroll
                        for (int j = 0; j < FN; ++j) q[j] = acc[i][j][v];
                    }
                    *reinterpret_cast<typename Group<FN>::type*>(C + (int64_t)m * N + fb.row(0, lane & 15)) = q;
                }
            }
        return;
    }
    if constexpr (WK > 1) {
        const int64_t tile = ((int64_t)entry * tiles_m + tm) * tiles_n + tn;
        double* mine = part + tile * slices * (NF * 256);
        if (wave == 0) {
#pragma unroll
            for (int f = 0; f < NF; ++f)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    ch::publish(mine + ((int64_t)z * NF + f) * 256 + v * 64 + lane, acc[f / FN][f % FN][v]);
        }
        if (!ch::last_block(&g_counters[tile], (uint32_t)slices)) return;
        constexpr int kFoldLoads = 4;  // slices in flight
        for (int f = wave; f < NF; f += 4) {
            double s[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) s[v] = ch::fetch(mine + (int64_t)f * 256 + v * 64 + lane);
            for (int q0 = 1; q0 < slices; q0 += kFoldLoads) {
                double x[kFoldLoads][4];
#pragma unroll
                for (int u = 0; u < kFoldLoads; ++u) {
                    const int q = min(q0 + u, slices - 1);
#pragma unroll
                    for (int v = 0; v < 4; ++v) x[u][v] = ch::fetch(mine + ((int64_t)q * NF + f) * 256 + v * 64 + lane);
                }
#pragma unroll
                for (int u = 0; u < kFoldLoads; ++u)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (q0 + u < slices) s[v] += x[u][v];
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) put(f, v, s[v]);
        }
    }
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// One product or batch as a kernel takes it.
struct Args {
    const double *a, *b;
    double* c;
    int M, N, K, batch;
    int64_t lda, ldb;  // row pitches of a and b as stored
};

int64_t tile_count(const Args& g, int tm, int tn) {
    return (int64_t)((g.M + tm - 1) / tm) * ((g.N + tn - 1) / tn) * g.batch;
}

template <bool KCA, bool KCB, bool V2A, bool V2B, int FM, int FN, int WK, int PF, int STEP>
int32_t launch(const Args& g, int slices) {
    constexpr int TM = 16 * FM * (WK == 1 ? 2 : 1), TN = 16 * FN * (WK == 1 ? 2 : 1);
    const int64_t tiles = tile_count(g, TM, TN);
    int64_t kslice = g.K;
    double* part = nullptr;
    if (slices > 1) {
        kslice = (((int64_t)g.K + slices - 1) / slices + STEP - 1) / STEP * STEP;
        slices = (int)((g.K + kslice - 1) / kslice);
        part = (double*)ch::scratch_try(11, sizeof(double) * (size_t)(tiles * slices * FM * FN * 256));
        if (!part) slices = 1, kslice = g.K;  // no room: K in one piece
    }
    gemm_f64_kernel<KCA, KCB, V2A, V2B, FM, FN, WK, PF, STEP><<<(unsigned)(tiles * slices), kThreads, 0, ch::stream()>>>(
        g.a, g.b, g.c, g.M, g.N, g.K, g.lda, g.ldb, (int64_t)g.M * g.K, (int64_t)g.K * g.N, (int64_t)g.M * g.N,
        (g.M + TM - 1) / TM, (g.N + TN - 1) / TN, g.batch, slices, kslice, part);
    CH_LAUNCHED("gemm_f64_kernel");
    return CLEAVE_HIP_OK;
}

// The wave tiles, and the time of a product on each as fitted to sweeps on
// MI355X (48 shapes and layouts from 33 x 77 x 1000 to 4096^3, and 26 outputs
// with K of 128 and 256; within 19% of the best of all measured):
//   base + max(busiest CU's MFMA time / eff + ends, one wave's steps x (MFMA + lat)) + fold
// A step, 16 of K here, is FM FN x 256 cycles of MFMA, 0.107 us a fragment pair.
// lat is what a wave's load latency adds where nothing else runs on its SIMD;
// ends, where K is up to 256, is the add of the partial tiles in LDS, by one wave, of
// each workgroup on a CU after the first: without it 20000 x 500 x 128 took 85 us on
// the 64 x 32 tiles, 62 on the 128 x 128 ones.
// eff_k applies where both operands are k-contiguous (A.B^T), whose 64-byte
// row pieces use the L1 less well.  Past one slice, each partial tile is
// written and read past the L2: about 3 TB/s for the two, and 3 us.
struct TileCost {
    int fm, fn, wk;
    double base, eff, eff_k, lat, end;  // us, share of the MFMA rate, us a step, us a tile
};
constexpr TileCost kTiles[] = {
    {1, 1, 4, 3.5, 0.32, 0.27, 0.3, 0.2},
    {2, 2, 4, 4.0, 0.65, 0.53, 0.6, 0.4},
    {4, 2, 4, 6.0, 0.77, 0.70, 0.6, 0.8},
    {4, 4, 1, 9.0, 0.86, 0.80, 0.6, 0.0},
};
constexpr int kSlices[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64};

struct Plan {
    int tile = 0, slices = 1;
};

Plan choose_tile(const Args& g, bool kca, bool kcb) {
    const bool both_k = kca && kcb;
    Plan best;
    double best_us = 1e300;
    const int cus = ch::num_cus();
    for (int i = 0; i < 4; ++i) {
        const TileCost& t = kTiles[i];
        const int tm = 16 * t.fm * (t.wk == 1 ? 2 : 1), tn = 16 * t.fn * (t.wk == 1 ? 2 : 1);
        const int64_t tiles = tile_count(g, tm, tn);
        if ((!kca && g.M < t.fm) || (!kcb && g.N < t.fn)) continue;  // a lane's group of rows must exist
        if (tiles > ch::kMaxBlocks) continue;  // run_matmul_f64 sees to it that some tile fits
        double last = 1e300;
        for (const int s : kSlices) {
            // slices of at least 128, at most 16 workgroups a CU, a counter per tile
            if (s > 1 && (t.wk == 1 || g.K / s < 128 || tiles * s > 16 * (int64_t)cus || tiles > kCounters)) break;
            const double steps = (double)((((int64_t)g.K + s - 1) / s + 16 * t.wk - 1) / (16 * t.wk));
            const double mfma = 0.107 * t.fm * t.fn;
            const double busiest = (double)((tiles * s + cus - 1) / cus);
            const double ends = g.K <= 256 ? (busiest - 1) * t.end : 0.0;
            const double busy = busiest * steps * mfma / (both_k ? t.eff_k : t.eff) + ends;
            const double chain = steps * (mfma + t.lat);
            const double us = t.base + (busy > chain ? busy : chain) +
                              (s > 1 ? 3.0 + (double)(tiles * s) * tm * tn * 16.0 / 3e6 : 0.0);
            if (us < best_us) best_us = us, best.tile = i, best.slices = s;
            if (us > last) break;  // more slices only add to the fold
            last = us;
        }
    }
    return best;
}

// Narrow products (M or N up to 16) stream the wide operand: 32 x 16 wave tiles
// (FM = 2, FN = 1, or the other way round), with as many slices as give every CU
// a workgroup while each keeps 256 of K, and on to four a CU while each keeps
// 1024.  8192 x 1 x 16384 188 us (5.7 TB/s) with 4 slices, 246 with one; 8192 x
// 16 x 1024 14.5 us with one, 15.5 with 2 or 4; 300 x 2 x 5000 36 with one, 9.8
// with 8.  The 64 x 16 tiles were level or slower on all of them.
int narrow_slices(const Args& g, int64_t tiles) {
    const int64_t cus = ch::num_cus();
    if (tiles > kCounters) return 1;
    int64_t s = (cus + tiles - 1) / tiles;
    if (s > g.K / 256) s = g.K / 256;
    int64_t more = 4 * cus / tiles;
    if (more > g.K / 1024) more = g.K / 1024;
    if (s < more) s = more;
    if (s > 64) s = 64;
    return s < 1 ? 1 : (int)s;
}

// Shallow products (K up to 64) of more than two and a half 64 x 64 tiles a CU
// mostly write C: waves on tiles of their own, four workgroups a CU.  Quarters of
// so short a K, and the 128 x 128 tiles' two workgroups a CU, left the stores
// uncovered (us): 65536 x 100 x 64 50 -> 29, 4096^2 x 8 34 -> 23, 256 of 128^2 x
// 64 23.6 -> 17.2, 2654 x 1520 x 3 12.8 -> 8.6.  Not where C fills under two thirds
// of the tiles (4096 of 32^2 x 32 18.5 on 16 x 16 tiles, 29 here), nor past K = 8
// with an odd N, whose rows the wider tiles store better (43 of 4031 x 267 x 16 104
// against 117).  A.B^T keeps the 128 x 128 tiles past K = 8, where C fills them:
// 4096^2 x 64 53 there, 67 here.
bool shallow(const Args& g, bool both_k) {
    const int64_t t64 = tile_count(g, 64, 64), t128 = tile_count(g, 128, 128);
    if (g.K > 64 || 2 * t64 <= 5 * (int64_t)ch::num_cus() || t64 > ch::kMaxBlocks) return false;
    if (2.0 * 64 * 64 * t64 > 3.0 * g.M * g.N * g.batch || (g.K > 8 && g.N % 2)) return false;
    return !both_k || g.K <= 8 || t128 < ch::num_cus() || t64 < 3 * t128;
}

template <bool KCA, bool KCB, bool V2A, bool V2B>
int32_t run_shape(const Args& g) {
    if (g.N <= 16 && (KCA || g.M >= 2))
        return launch<KCA, KCB, V2A, V2B, 2, 1, 4, 2, 16>(g, narrow_slices(g, tile_count(g, 32, 16)));
    if (g.M <= 16 && (KCB || g.N >= 2))
        return launch<KCA, KCB, V2A, V2B, 1, 2, 4, 2, 16>(g, narrow_slices(g, tile_count(g, 16, 32)));
    if ((KCA || g.M >= 2) && (KCB || g.N >= 2) && shallow(g, KCA && KCB))
        return launch<KCA, KCB, V2A, V2B, 2, 2, 1, 2, 8>(g, 1);
    const Plan p = choose_tile(g, KCA, KCB);
    switch (p.tile) {
        case 0: return launch<KCA, KCB, V2A, V2B, 1, 1, 4, 4, 16>(g, p.slices);
        case 1: return launch<KCA, KCB, V2A, V2B, 2, 2, 4, 1, 16>(g, p.slices);
        // Two k-contiguous operands whose rows are not 16-byte aligned load 8 bytes at a time,
        // and do better a whole step of 16 ahead: 1001^3 41 us against 45.5, 3001^3 973 against
        // 1164, 784 x 500 x 9999 177 against 211; aligned, 1000^3 40.5 against 41, 1200^3 108
        // against 83, and A.B 1000^3 44 against 39.
        case 2:
            if constexpr (KCA && KCB && !(V2A && V2B)) return launch<KCA, KCB, V2A, V2B, 4, 2, 4, 1, 16>(g, p.slices);
            else return launch<KCA, KCB, V2A, V2B, 4, 2, 4, 3, 8>(g, p.slices);
    }
    // A step ahead of 16 leaves the loads to the CU's other wave: 4096^3 A.B
    // 1906 us against 2190 with three of 8, 2000^3 274 against 268.
    if constexpr (!KCA || !KCB) return launch<KCA, KCB, V2A, V2B, 4, 4, 1, 1, 16>(g, 1);
    // Of two k-contiguous operands, aligned or not: up to K = 128 two steps of 8
    // ahead on two waves a SIMD, then three on one.  4096^2 x 64 53 us against 61,
    // 20000 x 500 x 128 71 against 70, x 256 142 against 119, 2000^3 276 against
    // 268 (4096^3 2101 against 2228; one of 16 on two waves 2181, 2000^3 303).
    else if (g.K <= 128) return launch<KCA, KCB, V2A, V2B, 4, 4, 1, 2, 8>(g, 1);
    else return launch<KCA, KCB, V2A, V2B, 4, 4, 1, 3, 8>(g, 1);
}

template <bool KCA, bool KCB>
int32_t run_layout(const Args& g) {
    // 16-byte loads along K need every row to start 16-byte aligned.
    const bool va = KCA && g.K % 2 == 0 && aligned16(g.a), vb = KCB && g.K % 2 == 0 && aligned16(g.b);
    if (va && vb) return run_shape<KCA, KCB, KCA, KCB>(g);
    if (va) return run_shape<KCA, KCB, KCA, false>(g);
    if (vb) return run_shape<KCA, KCB, false, KCB>(g);
    return run_shape<KCA, KCB, false, false>(g);
}

int32_t run_matmul_f64(const char* fn, const double* a, int64_t alen, const double* b, int64_t blen, double* c,
                       int64_t clen, int32_t batch, int32_t M, int32_t N, int32_t K, int32_t trans_a,
                       int32_t trans_b) {
    CH_REQUIRE(batch >= 1 && M >= 0 && N >= 0 && K >= 0, "%s: bad shape (batch %d, M %d, N %d, K %d)", fn, batch, M,
               N, K);
    CH_REQUIRE((trans_a == 0 || trans_a == 1) && (trans_b == 0 || trans_b == 1), "%s: trans flags must be 0 or 1",
               fn);
    const int64_t na = ch::count3(batch, M, K), nb = ch::count3(batch, K, N), nc = ch::count3(batch, M, N);
    CH_REQUIRE(na >= 0 && nb >= 0 && nc >= 0 && alen == na && blen == nb && clen == nc,
               "%s: lengths (%lld, %lld, %lld) do not match batch %d of %d x %d x %d", fn, (long long)alen,
               (long long)blen, (long long)clen, batch, M, N, K);
    if (clen == 0) return CLEAVE_HIP_OK;
    CH_REQUIRE(c && (K == 0 || (a && b)), "%s: null buffer", fn);
    CH_INIT_OR_RETURN();
    if (K > 0) {
        CH_DEVICE(fn, a, alen * 8);
        CH_DEVICE(fn, b, blen * 8);
    }
    CH_DEVICE(fn, c, clen * 8);
    // What fits a launch on the smallest tiles (16 x 16): `entries` of the batch, or, of one
    // narrow product (the others have larger tiles), a run of rows or of one row's columns.
    Args g{a, b, c, M, N, K, batch, trans_a ? M : K, trans_b ? K : N};
    auto run = [&]() {
        if (!trans_a && !trans_b) return run_layout<true, false>(g);
        if (!trans_a) return run_layout<true, true>(g);
        if (!trans_b) return run_layout<false, false>(g);
        return run_layout<false, true>(g);
    };
    if (tile_count(g, 16, 16) <= ch::kMaxBlocks) return run();
    g.batch = 1;
    const int64_t per = tile_count(g, 16, 16), entries = std::max<int64_t>(1, ch::kMaxBlocks / per);
    const int64_t most = ch::kMaxBlocks * 16;
    int64_t rows = M, cols = N;
    if (per > ch::kMaxBlocks && N <= 16) rows = most;
    else if (per > ch::kMaxBlocks && M <= 16) rows = 1, cols = most;
    for (int64_t e = 0; e < batch; e += entries)
        for (int64_t m = 0; m < M; m += rows)
            for (int64_t n = 0; n < N; n += cols) {
                g.batch = (int)std::min<int64_t>(entries, batch - e);
                g.M = (int)std::min<int64_t>(rows, M - m);
                g.N = (int)std::min<int64_t>(cols, N - n);
                g.a = a + e * M * K + (trans_a ? m : m * K);
                g.b = b + e * K * N + (trans_b ? n * K : n);
                g.c = c + e * M * N + m * N + n;
                const int32_t st = run();
                if (st != CLEAVE_HIP_OK) return st;
            }
    return CLEAVE_HIP_OK;
}

}  // namespace

extern "C" {

int32_t cleave_hip_matmul_f64(const double* a, int64_t alen, const double* b, int64_t blen, double* c, int64_t clen,
                              int32_t M, int32_t N, int32_t K, int32_t trans_a, int32_t trans_b) {
    return run_matmul_f64("cleave_hip_matmul_f64", a, alen, b, blen, c, clen, 1, M, N, K, trans_a, trans_b);
}

int32_t cleave_hip_matmul_batched_f64(const double* a, int64_t alen, const double* b, int64_t blen, double* c,
                                      int64_t clen, int32_t batch, int32_t M, int32_t N, int32_t K, int32_t trans_a,
                                      int32_t trans_b) {
    return run_matmul_f64("cleave_hip_matmul_batched_f64", a, alen, b, blen, c, clen, batch, M, N, K, trans_a,
                          trans_b);
}

}  // extern "C"
