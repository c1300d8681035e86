// Products of few rows against a matrix that is streamed once: every wave keeps a ring of slabs of its own in shared memory.  Shared by the plain products
// (gemm.hip) and the products over groups of rows (experts.hip).
#pragma once
#include "direct_tile.h"

// A work-group of four waves owns 8 WJ weight rows and all rows of x (8 XH at most).  K is dealt to its waves in slabs of 64 columns, slab s to wave s % 4; a wave
// requests its slabs (the weight rows' and x's 128 bytes each) straight into its own part of shared memory, D of them ahead, waits for its own requests alone and
// takes the products of a slab when it is there.  No barrier until the end, where the waves' sums meet in shared memory.
//
// Such a product takes as long as a compute unit needs to draw its share of the weights and its copy of x, and it draws at the rate of what it has on its way: a kernel
// whose waves fetch weight rows into registers (two steps of K each) behind a copy of x into shared memory had 16 to 32 KB on their way, fetched with sixteen rows to an
// instruction, and waited for x before the first product.  Here it is 4 D (WJ + XH) KB a work-group: 32 (one request of weights, up to 8 rows of x) to 80, up to which two work-groups
// fit a unit, and with 32 or 64 rows of x up to 128.  Each instruction fetches eight whole lines, and x arrives beside the weights.  Measured against that kernel (us, launch included,
// weights from memory; rows of x, N x K):
//   1 row: 2048 x 2048 3.8 -> 3.2, 4608 x 3584 8.1 -> 7.4;  8 rows: 256 x 2048 4.1 -> 3.1, 2048 x 2048 5.0 -> 3.5, 6144 x 2048 9.1 -> 6.5, 4096 x 4096 11.8 -> 7.6, gate and up
//   of 2 x 18944 x 3584 50.6 -> 46.9;  16 rows: 34 x 4096 8.9 -> 4.2, 2048 x 2048 6.2 -> 3.7, gate and up of 2 x 11264 x 4096 38.9 -> 32.0;  32 rows: 4608 x 3584 21.8 -> 10.8
//
// float: a slab is 32 columns, the same 128 bytes of every row, and the products are v_mfma_f32_16x16x4_f32's, which multiply and add in 32 bits.  A slab's sums are taken two instructions at a
// time from zero and then added to the wave's, so that a long sum has few roundings in a row.  An instruction takes 32 cycles, 256 a slab and block of weight rows: work-groups of few
// weight rows, which have a unit to themselves, deal K to eight waves; sum s % 8 of slab s is then a wave's only one, so the order is the same.
//
// HALVES 2: the weight rows are two halves of 4 WJ rows (the gate's and the up matrix's rows of the same outputs).
template <int WJ, typename T>
constexpr int ring_waves() { return sizeof(T) == 4 && WJ <= 3 ? 8 : 4; }
template <int WJ, int XH, int HALVES = 1, typename T = bf16_t>
struct RingShape {
    static constexpr int NW = ring_waves<WJ, T>();
    static constexpr int SLOT = (WJ + XH) * 1024;                          // bytes of a slab: 8 (WJ + XH) rows of 128
    static constexpr int FIT = 80 * 1024 / (NW * SLOT), D = FIT < 2 ? 2 : FIT > 4 ? 4 : FIT;
    static constexpr int HR = 8 * WJ / HALVES, SH = (HR + 15) / 16;        // weight rows of a half, and the blocks of 16 they make
    static constexpr int STRIPS = HALVES * SH, MT = (XH + 1) / 2;          // blocks of 16 weight rows and of 16 rows of x
    static constexpr int SETS = XH <= 2 ? 8 / NW : 1;                           // sets of sums a wave keeps: see ring_products
    static constexpr size_t LDS = (size_t)NW * D * SLOT;
    static_assert(8 * WJ % HALVES == 0 && (HALVES - 1) * HR + 16 * SH <= 8 * (WJ + XH), "a block that is not full reads on in its own slab");
    static_assert(SETS * STRIPS * MT * 1024 <= D * SLOT, "a wave's sums fit its own ring");
    static_assert((WJ + XH) * (D - 1) < 64 && LDS <= 160 * 1024, "requests on their way fit the counter, rings the shared memory");
};

// The products of `slabs` slabs: request j of a slab fetches eight rows of 128 bytes at w + woff[j] (x + xoff[j]), bytes, moved on by 128 a slab.  `wave` is uniform.
// On return every wave's sums lie in its ring (see ring_sum) and all waves have met.
//
// Up to 16 rows of x a product's numbers are summed in one order, whatever their number: slab s belongs to sum s % 8, so a wave keeps two sets, and lane group g holds the columns 16 g .. + 15 of a
// slab.  gemm_skinny_kernel with eight waves along K sums the same way, to the bit: the query/key/value projection of one row that makes its norm itself runs there, and a request must not notice
// which of the two served it.  With more rows a wave keeps one set.
//
// `spread`: the weight rows lie a multiple of 4 KB apart.  Work-groups in step then ask the same few channels of the memory for all their rows, so they begin at different slabs (see ring_start) and
// take them in turn from there.  The order of a sum then hangs on which work-group has the output, so up to 16 rows plan_ring deals such a product out alike whatever their number, and that
// projection does as it says (the gate of one row that makes its norm itself goes in step and is equal to rounding there: in these orders 18944 x 4096 took 70 us instead of 62).
// (us, in step -> spread: 16 rows, 8144 x 4096 16.3 -> 13.7, 32000 x 4096 48 -> 41, 4096 x 16384 33 -> 22, 11264 x 2048 10.9 -> 9.9; with other pitches, 4608 x 3584 8.1 -> 8.5, 2048 x 5632
// 8.4 -> 8.4.  Ranges of 512 columns in four orders, summed by pairs so that it would not hang on the work-group: 8144 x 4096 16.1, 4096 x 16384 34.  With few slabs a wave has them all on their
// way from the start, and 4096 columns by 1024 of K took 8.3 instead of 7.6.)
// Where a work-group begins: with up to 16 slabs a wave at 5 b + b / 8, beyond an eighth of the way on from its neighbour, which runs on the next XCD, and every eighth three slabs on.  With many
// slabs the first rule falls in with the pitch of the work-groups' rows at some sizes (us, first / second / the kernel that fetches into registers: 20000 x 8192, one row, 67.7 / 58.6 / 60.4,
// 10240 x 8192, 2 rows, 37.7 / 31.8 / 34.8, gate 24640 x 8192, 4 rows, 160 / 139 / 147; over 44 sizes of K 8192 and more the second takes 0.98 of the first), with few it is a little ahead
// (2560 x 2048, 16 rows, 4.5 / 4.7; over 22 sizes of K up to 4096 and up to 6144 columns 0.996).
template <typename T = bf16_t>
__host__ __device__ inline bool ring_spread(int pitch) { return pitch % (4096 / (int)sizeof(T)) == 0; }
__device__ __forceinline__ int ring_start(unsigned group, unsigned slabs_of_a_wave) {
    return (int)((slabs_of_a_wave <= 16 ? 5 * group + group / 8 : group % 8 * slabs_of_a_wave / 8 + 3 * (group / 8)) % slabs_of_a_wave);
}

template <int WJ, int XH, int HALVES, typename T>
__device__ __forceinline__ void ring_products(const T* w, const unsigned (&woff)[WJ], const T* x, const unsigned (&xoff)[XH], int slabs, char* ring, int wave, bool spread) {
    using S = RingShape<WJ, XH, HALVES, T>;
    constexpr int NW = S::NW, D = S::D, LPS = WJ + XH, MT = S::MT, COLS = 128 / sizeof(T);
    const int lane = threadIdx.x & 63, li = lane & 15, kg = lane >> 4;
    char* own = ring + wave * (D * S::SLOT);
    const unsigned own_at = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)((void __attribute__((address_space(3)))*)own));
    const int mine = slabs > wave ? (slabs - wave + NW - 1) / NW : 0;
    const int from = spread && mine >= 8 ? ring_start(blockIdx.x, mine) : 0;
    auto request = [&](int i) {
        const int turned = i + from < mine ? i + from : i + from - mine;
        const int k = COLS * (wave + turned * NW);
        const unsigned at = own_at + (unsigned)((i % D) * S::SLOT);
#pragma unroll
        for (int j = 0; j < WJ; ++j) load_to_lds_at(w + k, woff[j], at + j * 1024);
#pragma unroll
        for (int j = 0; j < XH; ++j) load_to_lds_at(x + k, xoff[j], at + (WJ + j) * 1024);
    };
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (d < mine) request(d);
    // where this lane's two pieces of a block lie in a slab
    int wat[S::STRIPS][2], xat[MT][2];
#pragma unroll
    for (int s = 0; s < S::STRIPS; ++s) {
        const int row = (s / S::SH) * S::HR + (s % S::SH) * 16 + li;
#pragma unroll
        for (int h = 0; h < 2; ++h) wat[s][h] = row * 128 + (((2 * kg + h) ^ ((row >> 1) & 7)) * 16);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int row = 8 * WJ + 16 * t + (XH == 1 ? li & 7 : li);
#pragma unroll
        for (int h = 0; h < 2; ++h) xat[t][h] = row * 128 + (((2 * kg + h) ^ ((row >> 1) & 7)) * 16);
    }
    f32x4_t acc[S::SETS][S::STRIPS][MT];
#pragma unroll
    for (int u = 0; u < S::SETS; ++u)
#pragma unroll
        for (int s = 0; s < S::STRIPS; ++s)
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[u][s][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto products = [&](int i, f32x4_t (&sums)[S::STRIPS][MT]) {
        const int after = mine - 1 - i;                 // slabs requested behind this one: D - 1 at most
        if (after >= D - 1) wait_direct_loads<(D - 1) * LPS>();
        else if (D > 3 && after == 2) wait_direct_loads<(D > 3 ? 2 : 0) * LPS>();
        else if (D > 2 && after == 1) wait_direct_loads<(D > 2 ? 1 : 0) * LPS>();
        else wait_direct_loads<0>();
        const char* slab = own + (i % D) * S::SLOT;
        f32x4_t part[2][2][S::STRIPS][MT];          // (float) a slab's sums by pairs of instructions
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            Frag16 wf[S::STRIPS], xf[MT];
#pragma unroll
            for (int t = 0; t < MT; ++t) xf[t].u = *(const uint4*)(slab + xat[t][h]);
#pragma unroll
            for (int s = 0; s < S::STRIPS; ++s) wf[s].u = *(const uint4*)(slab + wat[s][h]);
            if constexpr (sizeof(T) == 4) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int s = 0; s < S::STRIPS; ++s)
#pragma unroll
                        for (int t = 0; t < MT; ++t)
                            part[h][e & 1][s][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[s].f[e], xf[t].f[e], e < 2 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : part[h][e & 1][s][t], 0, 0, 0);
            } else {
#pragma unroll
                for (int s = 0; s < S::STRIPS; ++s)
#pragma unroll
                    for (int t = 0; t < MT; ++t) sums[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[s].v, xf[t].v, sums[s][t], 0, 0, 0);
            }
        }
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int s = 0; s < S::STRIPS; ++s)
#pragma unroll
                for (int t = 0; t < MT; ++t) sums[s][t] += (part[0][0][s][t] + part[0][1][s][t]) + (part[1][0][s][t] + part[1][1][s][t]);
        }
        if (i + D < mine) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // this slab has been read: its place is filled anew
            request(i + D);
        }
    };
    // (the last slab of an odd number stands behind the loop, not in it: with a way out between the two sets the compiler copied a set's registers from pass to pass, and
    // read one of them before the matrix instruction that writes it was through)
    int i = 0;
    for (; i + S::SETS <= mine; i += S::SETS) {
        products(i, acc[0]);
        if constexpr (S::SETS == 2) products(i + 1, acc[1]);
    }
    if (S::SETS == 2 && i < mine) products(i, acc[0]);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_nop 15" ::: "memory");      // (and the last products through, whichever way led here)
#pragma unroll
    for (int u = 0; u < S::SETS; ++u)
#pragma unroll
        for (int s = 0; s < S::STRIPS; ++s)
#pragma unroll
            for (int t = 0; t < MT; ++t) *(f32x4_t*)(own + ((u * S::STRIPS + s) * MT + t) * 1024 + lane * 16) = acc[u][s][t];
    __syncthreads();
}

// The waves' sums of block s of weight rows and block t of x: element v is weight row 16 (s % SH) + 4 (lane / 16) + v of half s / SH against x row 16 t + lane % 16.
template <int WJ, int XH, int HALVES, typename T = bf16_t>
__device__ __forceinline__ f32x4_t ring_sum(const char* ring, int s, int t) {
    using S = RingShape<WJ, XH, HALVES, T>;
    f32x4_t sum = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < S::SETS; ++u)
#pragma unroll
        for (int v = 0; v < S::NW; ++v) sum += *(const f32x4_t*)(ring + v * (S::D * S::SLOT) + ((u * S::STRIPS + s) * S::MT + t) * 1024 + (threadIdx.x & 63) * 16);
    return sum;
}

// The shapes that are built, and how outputs are dealt out: `wj` of the shape, `rows` outputs to a work-group (8 wj / halves at most).
struct RingPlan {
    int wj, rows;
};

// `units` compute units share `total` outputs: the shape with the least of (rounds of work-groups) x (requests of a work-group's weights, half of x's, which other work-groups have fetched into
// the caches as well, and a third of one for its start and end), then equal shares for all work-groups of these rounds: a launch is as slow as its busiest unit (4608 rows at 18 a unit 8.0 us, at
// 24 8.6, at 16 and two rounds 9.3).  No fewer than eight rows: one request fetches as many.
// A shape of six or eight requests has two slabs on its way, 56 to 80 KB, and with one work-group a unit that is all.  Up to 16 rows of x, where eight requests would fill a unit, two work-groups
// of four share it with 144 or 160 KB on their way; up to 8 rows of x also in a gate's place of six (us, one row: 16384 x 768 7.0 -> 6.7, x 2048 15.5 -> 13.6; gates, two rows: 8192 x 768
// 7.7 -> 7.1, x 3584 23.0 -> 22.4, 5120 x 768 5.7 -> 5.6; 16 rows, 5120 x 3584 15.5 -> 16.3, 8192 x 3584 22.9 -> 22.5).
// Not where K is split over work-groups (8 rows, one of eight / two of four, each 56 to 64 outputs of one range of K: 4096 x 4096 8.2 / 9.4, 3584 x 18944 25.3 / 26.6, 3072 x 8192 11.4 / 12.0,
// 5120 x 13824 28.0 / 28.2, 3584 x 3584 7.1 / 7.0).
// `spread` (see ring_products): up to 16 rows the same plan, that of 16.
// `pairs`: the float kernel's pairs of rows, which are built for three requests as well (4608 x 3584, 4 rows, 9 pairs to a work-group: 20.9 us in shapes of four requests, 18.4 of three).
static RingPlan plan_ring(int total, int M, int halves, int units, bool even, bool spread, bool split, bool pairs = false) {
    const int xh = M <= 8 && !spread ? 1 : M <= 16 ? 2 : M <= 32 ? 4 : 8, floor = 8 / halves;
    if (units < 1) units = 1;
    auto share = [&](long groups, long per) {
        int rows = (int)((total + groups - 1) / groups);
        if (even) rows += rows & 1;
        return rows < floor ? floor : rows > per ? (int)per : rows;
    };
    RingPlan best{0, 0};
    double least = 1e30;
    long best_rounds = 0;
    for (int wj : {1, 2, 3, 4, 6, 8}) {
        if (wj % halves && !(pairs && wj == 3)) continue;
        const long per = 8 * wj / halves, rounds = ((total + per - 1) / per + units - 1) / units;
        const double cost = rounds * (wj + 0.5 * xh + 0.3);
        if (cost >= least) continue;
        least = cost;
        best_rounds = rounds;
        best = RingPlan{wj, share(rounds * units, per)};
    }
    if (!split && best_rounds == 1 && (best.wj == 8 ? xh <= 2 : best.wj == 6 && xh == 1 && halves == 2)) best = RingPlan{4, share(2L * units, 32 / halves)};
    return best;
}
