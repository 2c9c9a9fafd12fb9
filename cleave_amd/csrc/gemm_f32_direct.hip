// gemm_f32_direct.hip -- f32 products with too few large tiles for the chip,
// on v_mfma_f32_16x16x4f32 without LDS staging.
//
// The LDS kernels (gemm_f32_tiled.hpp, gemm_f32_pingpong.hpp) want hundreds of
// 64 x 64 tiles or more.  Below that a wave computes a (16 FM) x (16 FN) tile
// of C from register fragments loaded straight from the caches, 16 of K at a
// time (FM FN x 128 cycles of MFMA a step), the other waves of its SIMD
// covering the loads.  A workgroup's four waves take quarters of K, added in
// LDS in wave order.  Past that K is cut into `slices` workgroups per tile;
// each publishes its partial tile and the last to arrive adds them in slice
// order (last_block.hpp).  The order of every sum depends on the shape alone.
//
// Every load is 16 bytes a lane (4 FM for an m/n-contiguous operand), whatever
// the alignment: global loads need 4-byte alignment only, so ragged rows need
// neither copies nor guards.
//   k-contiguous: over a 16-deep step, lane group h = lane / 16 takes k = 4h + s
//     at MFMA s, one load a fragment; fragment f holds rows 16 f + lane % 16.
//   m/n-contiguous: lane i = lane % 16 loads FM neighbouring rows at each of its
//     four k; fragment f holds row FM i + f.  A group that would pass the last
//     row starts FM rows before the end instead: it computes rows that its
//     neighbour has too, in the same order, and stores the same values.
// k past K enters as zero on both sides.
#include "common.hpp"
#include "gemm_common.hpp"
#include "last_block.hpp"

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));
template <int F>
struct Unaligned {
    typedef float type __attribute__((ext_vector_type(F), aligned(4)));
};
template <>
struct Unaligned<1> {
    typedef float type;
};

constexpr int kThreads = 256;
constexpr int kStep = 16;        // K per step of a wave
constexpr int kCounters = 4096;  // tiles that may be cut along K
static __device__ uint32_t g_counters[kCounters];  // 0 between launches

// One operand of a wave: F fragments of 16 rows (of A, or columns of B) by 16 of K.
template <int F, bool KC>
struct Frags {
    const float* p[KC ? F : 1];
    int64_t ld;
    int first, rows;

    __device__ __forceinline__ void init(const float* base, int64_t pitch, int r0, int nrows, int lane) {
        ld = pitch;
        first = r0;
        rows = nrows;
        const int h = lane >> 4, i = lane & 15;
        if constexpr (KC) {
#pragma unroll
            for (int f = 0; f < F; ++f) p[f] = base + (int64_t)min(r0 + 16 * f + i, nrows - 1) * pitch + 4 * h;
        } else {
            p[0] = base + (int64_t)(4 * h) * pitch + min(r0 + F * i, nrows - F);
        }
    }
    // The operand's row that fragment f holds at index i.
    __device__ __forceinline__ int row(int f, int i) const {
        return KC ? first + 16 * f + i : min(first + F * i, rows - F) + f;
    }
    __device__ __forceinline__ void load(int64_t k, float (&v)[F][4]) const {
        if constexpr (KC) {
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const typename Unaligned<4>::type x = *reinterpret_cast<const typename Unaligned<4>::type*>(p[f] + k);
#pragma unroll
                for (int s = 0; s < 4; ++s) v[f][s] = x[s];
            }
        } else {
#pragma unroll
            for (int s = 0; s < 4; ++s) take(p[0] + (k + s) * ld, s, v);
        }
    }
    // The step at k of a range that ends at k1 < k + 16.
    __device__ __forceinline__ void load_tail(int64_t k, int64_t k1, int lane, float (&v)[F][4]) const {
        const int h = lane >> 4;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const bool in = k + 4 * h + s < k1;
            if constexpr (KC) {
#pragma unroll
                for (int f = 0; f < F; ++f) v[f][s] = in ? p[f][k + s] : 0.0f;
            } else if (in) {
                take(p[0] + (k + s) * ld, s, v);
            } else {
#pragma unroll
                for (int f = 0; f < F; ++f) v[f][s] = 0.0f;
            }
        }
    }
    __device__ __forceinline__ static void take(const float* q, int s, float (&v)[F][4]) {
        if constexpr (F == 1) {
            v[0][s] = *q;
        } else {
            const typename Unaligned<F>::type x = *reinterpret_cast<const typename Unaligned<F>::type*>(q);
#pragma unroll
            for (int f = 0; f < F; ++f) v[f][s] = x[f];
        }
    }
};

// `part`: tiles x slices partial tiles, unused with slices == 1.  A 1-D grid of
// tiles_m * tiles_n * batch * slices workgroups.
template <bool KCA, bool KCB, int FM, int FN, int PF>
__global__ __launch_bounds__(kThreads) void gemm_f32_direct_kernel(
    const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C, int M, int N, int K, int64_t lda,
    int64_t ldb, int64_t sa, int64_t sb, int64_t sc, int tiles_m, int tiles_n, int batch, int slices, int64_t kslice,
    float* part) {
    constexpr int WK = 4, NF = FM * FN;  // waves along K; fragments
    __shared__ float red[(WK - 1) * NF * 4 * 64];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int b, tm, tn;  // b: batch entry and slice
    ch::block_coords(blockIdx.x, tiles_m, tiles_n, batch * slices, b, tm, tn);
    const int entry = b / slices, z = b - entry * slices;
    A += (int64_t)entry * sa;
    B += (int64_t)entry * sb;
    C += (int64_t)entry * sc;
    const int m0 = tm * 16 * FM, n0 = tn * 16 * FN;

    int64_t k0 = z * kslice, k1 = min((int64_t)K, k0 + kslice);
    {
        const int64_t steps = (k1 - k0 + kStep - 1) / kStep, each = (steps + WK - 1) / WK * kStep;
        k0 += wave * each;
        k1 = min(k1, k0 + each);
    }

    v4f acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    auto mfma = [&](const float (&a)[FM][4], const float (&bb)[FN][4]) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][s], bb[j][s], acc[i][j], 0, 0, 0);
    };

    Frags<FM, KCA> fa;
    Frags<FN, KCB> fb;
    fa.init(A, lda, m0, M, lane);
    fb.init(B, ldb, n0, N, lane);
    if (k0 < k1) {
        const int whole = (int)((k1 - k0) / kStep);
        float a[PF][FM][4], bb[PF][FN][4];
#pragma unroll
        for (int u = 0; u < PF; ++u)
            if (u < whole) {
                fa.load(k0 + u * kStep, a[u]);
                fb.load(k0 + u * kStep, bb[u]);
            }
        for (int t = 0; t < whole; t += PF) {
#pragma unroll
            for (int u = 0; u < PF; ++u)
                if (t + u < whole) {
                    mfma(a[u], bb[u]);
                    if (t + u + PF < whole) {
                        fa.load(k0 + (int64_t)(t + u + PF) * kStep, a[u]);
                        fb.load(k0 + (int64_t)(t + u + PF) * kStep, bb[u]);
                    }
                }
        }
        k0 += (int64_t)whole * kStep;
        if (k0 < k1) {
            fa.load_tail(k0, k1, lane, a[0]);
            fb.load_tail(k0, k1, lane, bb[0]);
            mfma(a[0], bb[0]);
        }
    }

    if (wave > 0) {
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int v = 0; v < 4; ++v) red[(((wave - 1) * NF + f) * 4 + v) * 64 + lane] = acc[f / FN][f % FN][v];
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int w = 0; w < WK - 1; ++w)
#pragma unroll
            for (int f = 0; f < NF; ++f)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[f / FN][f % FN][v] += red[((w * NF + f) * 4 + v) * 64 + lane];
    }

    // acc[i][j][v]: index 4 (lane / 16) + v of A's fragment i, lane % 16 of B's fragment j.
    auto put_row = [&](int i, int v, const float (&x)[FN]) {
        const int m = fa.row(i, 4 * (lane >> 4) + v);
        if (KCA && m >= M) return;
        float* c = C + (int64_t)m * N;
        if constexpr (KCB || FN == 1) {
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const int n = fb.row(j, lane & 15);
                if (n < N) c[n] = x[j];
            }
        } else {
            typename Unaligned<FN>::type q;
#pragma unroll
            for (int j = 0; j < FN; ++j) q[j] = x[j];
            *reinterpret_cast<typename Unaligned<FN>::type*>(c + fb.row(0, lane & 15)) = q;
        }
    };
    if (slices == 1) {
        if (wave != 0) return;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                float x[FN];
#pragma unroll
                for (int j = 0; j < FN; ++j) x[j] = acc[i][j][v];
                put_row(i, v, x);
            }
        return;
    }
    const int64_t tile = ((int64_t)entry * tiles_m + tm) * tiles_n + tn;
    v2f* mine = reinterpret_cast<v2f*>(part) + tile * slices * (NF * 128) + lane;
    if (wave == 0) {
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int q = 0; q < 2; ++q)
                ch::publish(mine + ((int64_t)z * NF + f) * 128 + q * 64,
                            v2f{acc[f / FN][f % FN][2 * q], acc[f / FN][f % FN][2 * q + 1]});
    }
    if (!ch::last_block(&g_counters[tile], (uint32_t)slices)) return;
    // wave w adds rows v = 2q, 2q + 1 of fragment rows i, (i, q) = w, w + 4, ...
    constexpr int kFoldLoads = FN >= 4 ? 2 : 4;  // slices in flight
    for (int g = wave; g < FM * 2; g += 4) {
        const int i = g >> 1, q = g & 1;
        v2f s[FN];
#pragma unroll
        for (int j = 0; j < FN; ++j) s[j] = ch::fetch(mine + (int64_t)(i * FN + j) * 128 + q * 64);
        for (int z0 = 1; z0 < slices; z0 += kFoldLoads) {
            v2f x[kFoldLoads][FN];
#pragma unroll
            for (int u = 0; u < kFoldLoads; ++u) {
                const int zz = min(z0 + u, slices - 1);
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    x[u][j] = ch::fetch(mine + ((int64_t)zz * NF + i * FN + j) * 128 + q * 64);
            }
#pragma unroll
            for (int u = 0; u < kFoldLoads; ++u)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    if (z0 + u < slices) {
                        s[j][0] += x[u][j][0];
                        s[j][1] += x[u][j][1];
                    }
        }
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            float x[FN];
#pragma unroll
            for (int j = 0; j < FN; ++j) x[j] = s[j][v];
            put_row(i, 2 * q + v, x);
        }
    }
}

struct Args {
    const float *a, *b;
    float* c;
    int M, N, K, batch;
};

int64_t tile_count(const Args& g, int tm, int tn) {
    return (int64_t)((g.M + tm - 1) / tm) * ((g.N + tn - 1) / tn) * g.batch;
}

template <bool KCA, bool KCB, int FM, int FN, int PF>
int32_t launch(const Args& g, int slices) {
    constexpr int TM = 16 * FM, TN = 16 * FN;
    const int64_t tiles = tile_count(g, TM, TN);
    int64_t kslice = g.K;
    float* part = nullptr;
    if (slices > 1) {
        kslice = (((int64_t)g.K + slices - 1) / slices + kStep - 1) / kStep * kStep;
        slices = (int)((g.K + kslice - 1) / kslice);
        part = (float*)ch::scratch_try(12, sizeof(float) * (size_t)(tiles * slices * FM * FN * 256));
        if (!part) slices = 1, kslice = g.K;  // no room: K in one piece
    }
    gemm_f32_direct_kernel<KCA, KCB, FM, FN, PF><<<(unsigned)(tiles * slices), kThreads, 0, ch::stream()>>>(
        g.a, g.b, g.c, g.M, g.N, g.K, KCA ? g.K : g.M, KCB ? g.K : g.N, (int64_t)g.M * g.K, (int64_t)g.K * g.N,
        (int64_t)g.M * g.N, (g.M + TM - 1) / TM, (g.N + TN - 1) / TN, g.batch, slices, kslice, part);
    CH_LAUNCHED("gemm_f32_direct_kernel");
    return CLEAVE_HIP_OK;
}

// The wave tiles, and the time of a product on each as fitted to sweeps on
// MI355X (39 shapes from 50 x 70 x 20 to 1500^3, all layouts):
//   base + max(busiest CU's MFMA time / eff, one wave's steps x (MFMA + lat)) + fold
// A step of a wave is FM FN x 128 cycles of MFMA, 0.0533 us a fragment pair.
// lat is what a wave's load latency adds where nothing else runs on its SIMD.
// Past one slice each partial tile is written and read past the L2, about 3
// TB/s for the two, and 2 us.  The 2:1 tile is turned to give an
// m/n-contiguous operand the wide side.
struct TileCost {
    int fm, fn;
    double base, eff, lat;  // us, share of the MFMA rate, us a step
};
constexpr TileCost kTiles[] = {
    {1, 1, 4.0, 0.30, 0.07},
    {2, 2, 4.0, 0.44, 0.16},
    {4, 2, 5.0, 0.60, 0.15},
    {4, 4, 7.0, 0.70, 0.30},
};
constexpr int kSlices[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64};

struct Plan {
    int tile = -1, slices = 1;
    double us = 1e300;
};

Plan choose_tile(const Args& g, bool kca, bool kcb) {
    Plan best;
    const int cus = ch::num_cus();
    for (int i = 0; i < 4; ++i) {
        const TileCost& t = kTiles[i];
        const int fm = i == 2 && !kcb ? t.fn : t.fm, fn = i == 2 && !kcb ? t.fm : t.fn;
        if ((!kca && g.M < fm) || (!kcb && g.N < fn)) continue;  // a lane's group of rows must exist
        const int64_t tiles = tile_count(g, 16 * fm, 16 * fn);
        if (tiles > 0x7FFFFFFF) continue;
        double last = 1e300;
        for (const int s : kSlices) {
            // slices of at least 128, at most 16 workgroups a CU, a counter per tile
            if (s > 1 && (g.K / s < 128 || tiles * s > 16 * (int64_t)cus || tiles > kCounters)) break;
            const double steps = (double)((((int64_t)g.K + s - 1) / s + kStep * 4 - 1) / (kStep * 4));
            const double mfma = 0.0533 * fm * fn;
            const double busy = (double)((tiles * s + cus - 1) / cus) * steps * mfma / t.eff;
            const double chain = steps * (mfma + t.lat);
            const double us = t.base + (busy > chain ? busy : chain) +
                              (s > 1 ? 2.0 + (double)(tiles * s) * fm * fn * 256 * 8.0 / 3e6 : 0.0);
            if (us < best.us) best.us = us, best.tile = i, best.slices = s;
            if (us > last) break;  // more slices only add to the fold
            last = us;
        }
    }
    return best;
}

template <bool KCA, bool KCB>
int32_t run_layout(const Args& g, const Plan& p) {
    switch (p.tile) {
        case 0: return launch<KCA, KCB, 1, 1, 4>(g, p.slices);
        case 1: return launch<KCA, KCB, 2, 2, 1>(g, p.slices);
        case 2: return launch<KCA, KCB, KCB ? 4 : 2, KCB ? 2 : 4, 1>(g, p.slices);
        default: return launch<KCA, KCB, 4, 4, 1>(g, p.slices);
    }
}

}  // namespace

namespace ch {
// Runs the product (or batch) on these tiles when they are expected to take
// under `most_us` microseconds; *st is the outcome.  False when not run.
bool try_direct_f32(const float* a, const float* b, float* c, int M, int N, int K, int batch, int ta, int tb,
                    double most_us, int32_t* st) {
    const Args g{a, b, c, M, N, K, batch};
    const Plan p = choose_tile(g, !ta, tb);
    if (p.tile < 0 || p.us >= most_us) return false;
    if (!ta && !tb) *st = run_layout<true, false>(g, p);
    else if (!ta) *st = run_layout<true, true>(g, p);
    else if (!tb) *st = run_layout<false, false>(g, p);
    else *st = run_layout<false, true>(g, p);
    return true;
}
}  // namespace ch
