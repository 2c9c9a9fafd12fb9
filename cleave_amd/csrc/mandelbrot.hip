// mandelbrot.hip -- escape-time map of examples/mandelbrot.cleave:14-26 in f32.
//
// escape_count(c): z = 0; for n in 0..max_iter { z = z*z + c;
// if |z|^2 > 4 { return n } }; return max_iter.  Complex mul/add and
// magnitude_sq follow stdlib/complex/complex.cleave:25-32 and :54:
//   re = zr*zr - zi*zi;  im = zr*zi + zi*zr;  z = (re + cr, im + ci);
//   |z|^2 = zr*zr + zi*zi.
// The reference latches the first escape and keeps iterating; this kernel
// does the same inside unrolled blocks of iterations and stops a wave once all
// of its lanes are decided: escaped, or back on a state they had before.
//
// z -> z*z + c is a function of (zr, zi) alone, in f32 as in exact arithmetic.
// A lane whose (zr, zi) equals an earlier pair repeats the iterations between
// the two for ever; none of them escaped, so its count is max_iter, the value
// the whole loop would return.  (Equal here is ==: a zero of the other sign
// gives the same |zr|, |zi| ever after, and NaN equals nothing and runs on.)
// Rounding makes the orbits inside the set fall onto such cycles: over
// [-2,1] x [-1.5,1.5] at 16384^2 x 1000 a wave's longest lane runs 64
// iterations on average instead of 189, and the map takes 2.26 ms instead of
// 5.64, bound by VALU issue as before; windows at the set's edge without such
// orbits take the same time (2112 x 968, span 0.024, 236 iterations: 22.7 us).
//
// Bit-exactness: the library is compiled with -ffp-contract=off, so no mul+add
// is fused behind the code's back.  Three rewrites are exact and save work:
//   * the zr*zr and zi*zi of the |z|^2 test are the same rounded products the
//     next step's re needs;
//   * zr*zi + zi*zr == p + p with p = fl(zr*zi) (the same rounded product
//     added to itself), and p + p == 2p exactly;
//   * so im + ci = fl(fl(2p) + ci) = fl(2p + ci) = fma(2, p, ci): 2p is exact
//     in binary floating point (subnormals included), so the fma's single
//     rounding is the two-step sum's second one.  Where 2p overflows, |ci|
//     is far below half an ulp of FLT_MAX and both forms give the same inf.
//
// Mapping: one wave per 8 x 8 pixel block (neighbouring pixels have similar
// iteration counts, so waves diverge less than with 64 x 1 strips); a
// 256-thread workgroup covers 16 x 16 pixels.
#include "common.hpp"

namespace {

// Iterations per block of the unrolled loop.  Inside a block every lane
// iterates, and the lanes still inside the radius after each iteration are
// kept as a wave mask (the escape compare writes a mask, a scalar AND narrows
// it).  A lane whose first escape is iteration n gets count n, and one that
// never escapes gets max_iter (the reference's `escaped`/`count` latch,
// examples/mandelbrot.cleave:14-26).  Per iteration: 7 arithmetic ops and a
// compare on the VALU, one scalar AND -- no branch, no count update.  Only in
// a block where some lane escapes are the escaping lanes' counts formed, from
// the block's masks: n = the block's first iteration + the number of the
// block's masks that still hold the lane, taken bit by bit from the masks with
// scalar operations (eight adds with carry took 2-4% more over small windows).
// The wave leaves once no lane is alive.  With 9 VALU per iteration (before 2p + ci became one fma), at
// 16384^2 x 1000 blocks of 8 measured 6.10 ms, blocks of 16 6.28 ms, and a
// count added every iteration 6.69 ms; on another box blocks of 4, 6, 8 and
// 12 measured 6.40, 6.19, 6.12 and 6.21 ms.  The fma form: 5.61 ms.
constexpr int kBlockIters = 8;

// The state each block's end is compared with is first taken after kFirstTake
// iterations, so a wave that is done by then pays nothing for it, and retaken
// each time the count has grown by half: the distance between takes grows, so
// cycles of any length fit in sooner or later, and at most half as many
// iterations again pass before a settled orbit is seen.  A block's end meets a
// cycle of p iterations lcm(p, kBlockIters) after the take.  Iterations of a
// wave's longest lane, on average over 6000 waves of the grid above and of a
// window at its edge, [-0.9, -0.6] x [-0.05, 0.25] at 4096^2: without 189 / 863;
// first after 16 63.7 / 409.9, 48 63.6 / 409.9, 96 66.9 / 412.5; takes at twice
// the count 64.6 / 423, every 64 iterations 82 / 501; blocks of 16, 82 / 473.
constexpr int kFirstTake = 48;

// if_set in the lanes set in `lanes`, if_clear in the others.
__device__ __forceinline__ uint32_t select_lanes(uint64_t lanes, uint32_t if_set, uint32_t if_clear) {
    uint32_t r;
    asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(r) : "v"(if_clear), "v"(if_set), "s"(lanes));
    return r;
}

// Bit (1, 2 or 4) in the lanes set in `lanes`, 0 in the others.
template <int Bit>
__device__ __forceinline__ uint32_t bit_lanes(uint64_t lanes) {
    uint32_t r;
    asm("v_cndmask_b32_e64 %0, 0, %1, %2" : "=v"(r) : "n"(Bit), "s"(lanes));
    return r;
}

__global__ __launch_bounds__(256) void mandelbrot_kernel(uint32_t* __restrict__ out, int width,
                                                         int height, float x0, float y0, float dx,
                                                         float dy, int max_iter) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = blockIdx.x * 16 + (wave & 1) * 8 + (lane & 7);
    const int row = blockIdx.y * 16 + (wave >> 1) * 8 + (lane >> 3);
    const bool inside = col < width && row < height;
    const float cr = x0 + (float)col * dx;
    const float ci = y0 + (float)row * dy;
    float zr = 0.0f, zi = 0.0f, zr2 = 0.0f, zi2 = 0.0f;
    uint32_t count = 0;  // final in the lanes that have escaped
    uint64_t alive = __builtin_amdgcn_ballot_w64(inside);
    uint64_t cycling = 0;  // lanes that have met the state kept
    int n = 0;
    // Whole blocks: lanes past their escape keep iterating (z may overflow to
    // inf/NaN, which no longer matters: the count is latched).
    auto block = [&]() {
        const uint64_t before = alive;
        uint64_t after[kBlockIters];  // alive after each iteration of the block
#pragma unroll
        for (int u = 0; u < kBlockIters; ++u) {
            const float p = zr * zi;
            const float re = zr2 - zi2;
            zr = re + cr;
            zi = __builtin_fmaf(2.0f, p, ci);  // (p + p) + ci, exactly
            zr2 = zr * zr;
            zi2 = zi * zi;
            alive &= __builtin_amdgcn_ballot_w64(!(zr2 + zi2 > 4.0f));
            after[u] = alive;
        }
        const uint64_t escaped = before & ~alive;
        if (escaped != 0) {  // wave-uniform
            // the number of the block's masks that still hold an escaped lane,
            // 0..7, bit by bit: each mask lies inside the one before
            const uint64_t b0 = (after[0] & ~after[1]) | (after[2] & ~after[3]) | (after[4] & ~after[5]) | after[6];
            const uint64_t b1 = (after[1] & ~after[3]) | after[5];
            const uint32_t c = (uint32_t)n + (bit_lanes<4>(after[3]) | bit_lanes<2>(b1) | bit_lanes<1>(b0));
            count = select_lanes(escaped, c, count);
        }
    };
    const int whole = max_iter & ~(kBlockIters - 1);
    // A wave with no lane left sets n to kDone: one loop condition, one exit.
    constexpr int kDone = 0x7FFFFFFF;
    uint32_t next_take = kFirstTake;
    int stop = whole < kFirstTake ? whole : kFirstTake;
    while (n < stop) {
        block();
        n = alive != 0 ? n + kBlockIters : kDone;
    }
    while (n < whole) {
        const float sr = zr, si = zi;  // the state that the next blocks' ends are compared with
        next_take += next_take / 2;
        stop = (uint32_t)whole < next_take ? whole : (int)next_take;
        while (n < stop) {
            block();
            uint64_t met = __builtin_amdgcn_ballot_w64(zr == sr) & alive;
            if (met != 0) {  // wave-uniform
                met &= __builtin_amdgcn_ballot_w64(zi == si);
                cycling |= met;
                alive &= ~met;
            }
            n = alive != 0 ? n + kBlockIters : kDone;
        }
    }
    // Remaining max_iter % kBlockIters iterations (only when some lane survived).
    for (int m = n; m < max_iter && alive != 0; ++m) {
        const uint64_t before = alive;
        const float p = zr * zi;
        const float re = zr2 - zi2;
        zr = re + cr;
        zi = __builtin_fmaf(2.0f, p, ci);
        zr2 = zr * zr;
        zi2 = zi * zi;
        alive &= __builtin_amdgcn_ballot_w64(!(zr2 + zi2 > 4.0f));
        count = select_lanes(before & ~alive, (uint32_t)m, count);
    }
    count = select_lanes(alive | cycling, (uint32_t)max_iter, count);  // never escaped
    if (inside) out[(int64_t)row * width + col] = count;
}

}  // namespace

extern "C" int32_t cleave_hip_mandelbrot_u32(uint32_t* out, int64_t outlen, int32_t width,
                                             int32_t height, float x0, float y0, float dx,
                                             float dy, int32_t max_iter) {
    CH_REQUIRE(width > 0 && height > 0, "cleave_hip_mandelbrot_u32: width/height must be positive");
    CH_REQUIRE(max_iter >= 0, "cleave_hip_mandelbrot_u32: max_iter must be >= 0");
    CH_REQUIRE(outlen == (int64_t)width * height, "cleave_hip_mandelbrot_u32: outlen %lld != width*height %lld",
               (long long)outlen, (long long)width * height);
    CH_REQUIRE(out != nullptr, "cleave_hip_mandelbrot_u32: null buffer");
    CH_INIT_OR_RETURN();
    CH_DEVICE("cleave_hip_mandelbrot_u32", out, outlen * 4);
    dim3 grid((unsigned)((width + 15) / 16), (unsigned)((height + 15) / 16));
    CH_REQUIRE(grid.y <= 65535u, "cleave_hip_mandelbrot_u32: height %d too large", height);
    mandelbrot_kernel<<<grid, 256, 0, ch::stream()>>>(out, width, height, x0, y0, dx, dy, max_iter);
    CH_LAUNCHED("mandelbrot_kernel");
    return CLEAVE_HIP_OK;
}
