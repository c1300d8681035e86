// The matrix product's tile kernel whose operands go straight into shared memory, shared by the plain products (gemm.hip) and the products
// over groups of rows (experts.hip), with the types that both use.
#pragma once
#include "activation.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

typedef float f32x16_t __attribute__((ext_vector_type(16)));

// Several products of equal shape in one launch (the mixes of a token and the one before it, each against its own matrix): product
// blockIdx.z reads x and w and writes out these many elements further on.
struct GroupStride {
    long x, w, out;
};
struct Groups {
    int count = 1;
    GroupStride stride{0, 0, 0};
};

union Frag16 {          // 16 bytes: eight bfloat16 as the MFMA wants them, or one 128-bit load
    uint4 u;
    bf16x8_t v;
    float f[4];
};

// The gate of a fused gate/up product: GATE 1: silu(g) * u, GATE 2: relu(g) * u, GATE 3: gelu(g) * u in its tanh form (the value of SW in the
// kernels below; 0: no gate).
template <int GATE>
__device__ __forceinline__ float gate_mul(float g, float u) { return (GATE == 3 ? gelu_tanh(g) : GATE == 2 ? fmaxf(g, 0.f) : g / (1.f + expf(-g))) * u; }

// Shared memory beyond 64 KB has to be allowed per kernel, once per process.
template <typename Kernel>
static hipError_t allow_lds(Kernel kernel, size_t bytes) {
    if (bytes <= 65536) return hipSuccess;
    return hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

// =====================================================================================
// The same product with the operands fetched straight into shared memory (K a multiple of 64).
//
// global_load_lds_dwordx4 moves 16 bytes per lane from memory into shared memory without passing
// through registers: one instruction of a wave fills 1 KB, eight rows of a 64-element slab.  A slab
// row is 128 bytes with no padding; piece c (16 bytes) of row r lies in slot c ^ ((r >> 1) & 7), so
// that the sixteen rows a quarter-wave reads for one MFMA operand fall on all 64 banks (measured:
// no bank conflicts).  The lane that fills slot s of row r therefore fetches piece s ^ ((r >> 1) & 7)
// of that row from memory.  STAGES slabs are in flight or in use: the slab STAGES - 1 ahead is
// requested into the buffer that a step has just finished with, and a step ends with a wait for
// this wave's requests of the next slab and one barrier.
// The requests are issued as assembly: the compiler orders every later shared-memory read behind
// a direct load it knows of (a full wait per slab), so the kernel keeps that order itself.  The
// address is a base that the wave shares and a 32-bit offset per lane.
__device__ __forceinline__ void load_to_lds_at(const void* base, unsigned offset, unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" :: "v"(offset), "s"(base), "s"(lds_addr) : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void wait_direct_loads() { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory"); }

// Rows of one slab in shared memory: the BM rows of x and the BN rows of w, rounded up to what the waves'
// load instructions (64 lanes x 16 bytes each) fill between them.
constexpr int dl_slab_rows(int bm, int bn, int waves) {
    const int per = 8 * waves;
    return (bm + bn + per - 1) / per * per;
}

// The result tile of a group of rows: the activation applied to the accumulators (PAIRS: to a lane's neighbouring columns 2i and 2i + 1, which give
// one output column), laid out row by row in the free slab buffers as below and stored in whole rows.
template <int ACT>
__device__ __forceinline__ float activated(float v) { return activate(v, ACT); }

template <int ACT, int BM, int BN, int WM, int WN, int FM, int FN, int ROOM, bool PAIRS>
__device__ __forceinline__ void store_expert_tile_as(const f32x4_t (&acc)[FM][FN], bf16_t* stage, bf16_t* out, int r0, int c0, int M, int N, int ldo) {
    constexpr int WNO = PAIRS ? WN / 2 : WN;
    static_assert(BM * (PAIRS ? BN / 2 : BN) <= ROOM, "the result tile must fit the slab buffers");
    const int lane = threadIdx.x & 63, lm = lane & 15, quad = lane >> 4;
    const int cols = PAIRS ? N / 2 : N, co = PAIRS ? c0 / 2 : c0;
    const bool whole = cols % 8 == 0 && ldo % 8 == 0 && ((uintptr_t)out % 16) == 0;
    constexpr int C = WNO / 8, CX = C & -C;
    static_assert((WM * C) % 64 == 0, "the rows of a wave tile must divide over its lanes");
    if (whole) __syncthreads();
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            constexpr int V = PAIRS ? 2 : 4;              // output columns of a lane's four
            bf16_t h[V];
#pragma unroll
            for (int e = 0; e < V; ++e) {
                if constexpr (PAIRS) h[e] = from_float<bf16_t>(activated<ACT>(acc[i][j][2 * e]) * acc[i][j][2 * e + 1]);
                else h[e] = from_float<bf16_t>(activated<ACT>(acc[i][j][e]));
            }
            const int n = (j * 16 + 4 * quad) / (PAIRS ? 2 : 1), row = i * 16 + lm;
            if (whole) {
                bf16_t* dst = stage + row * WNO + (((n >> 3) ^ (row & (CX - 1))) * 8) + (n & 7);
                const uint32_t a = (uint32_t)h[0].bits | ((uint32_t)h[1].bits << 16);
                if constexpr (PAIRS) *(uint32_t*)dst = a;
                else *(uint2*)dst = make_uint2(a, (uint32_t)h[V - 2].bits | ((uint32_t)h[V - 1].bits << 16));
            } else if (r0 + row < M) {
#pragma unroll
                for (int e = 0; e < V; ++e)
                    if (co + n + e < cols) out[(size_t)(r0 + row) * ldo + co + n + e] = h[e];
            }
        }
    if (!whole) return;
    // (one wave's shared-memory accesses are carried out in order: no wait in between)
#pragma unroll
    for (int q = 0; q < WM * C / 64; ++q) {
        const int idx = q * 64 + lane, row = idx / C, piece = idx % C;
        const uint4 val = *(const uint4*)(stage + row * WNO + ((piece ^ (row & (CX - 1))) * 8));
        if (r0 + row < M && co + piece * 8 < cols) *(uint4*)(out + (size_t)(r0 + row) * ldo + co + piece * 8) = val;
    }
}

template <int BM, int BN, int WM, int WN, int FM, int FN, int ROOM, bool PAIRS>
__device__ __forceinline__ void store_expert_tile(const f32x4_t (&acc)[FM][FN], bf16_t* stage, bf16_t* out, int r0, int c0, int M, int N, int ldo, int act) {
    switch (act & ~ACT_PAIRS) {         // (one switch for the tile, not one for every number)
    case ACT_RELU2: return store_expert_tile_as<ACT_RELU2, BM, BN, WM, WN, FM, FN, ROOM, PAIRS>(acc, stage, out, r0, c0, M, N, ldo);
    case ACT_SILU: return store_expert_tile_as<ACT_SILU, BM, BN, WM, WN, FM, FN, ROOM, PAIRS>(acc, stage, out, r0, c0, M, N, ldo);
    case ACT_GELU_TANH: return store_expert_tile_as<ACT_GELU_TANH, BM, BN, WM, WN, FM, FN, ROOM, PAIRS>(acc, stage, out, r0, c0, M, N, ldo);
    case ACT_GELU: return store_expert_tile_as<ACT_GELU, BM, BN, WM, WN, FM, FN, ROOM, PAIRS>(acc, stage, out, r0, c0, M, N, ldo);
    default: return store_expert_tile_as<ACT_NONE, BM, BN, WM, WN, FM, FN, ROOM, PAIRS>(acc, stage, out, r0, c0, M, N, ldo);
    }
}

// Groups of rows (GS = ExpertRows): group g owns the output rows offsets[g] .. offsets[g + 1] - 1 and the g-th of the matrices w [groups,
// N, K]; `src` (optional) maps an output row to the row of x it reads.  How many rows a group has is known on the GPU alone, so the grid is an
// upper bound: a work-group adds up the groups' tiles, finds its own among them and ends at once if there is none.  The tiles of a group follow
// each other, those that read the same weight rows side by side, and each XCD gets a stretch of them, so a group's matrix passes through one L2.
// Measured against a kernel whose waves fetch their operands from memory into registers: see pick_experts.
template <bool PAIRS_>
struct ExpertRows {
    static constexpr bool PAIRS = PAIRS_;      // the activation joins the columns 2i and 2i + 1 into one output column
    const int* offsets;
    const int* src;
    int groups, act;
};
template <typename GS> struct IsExpertRows { static constexpr bool value = false, pairs = false; };
template <bool P> struct IsExpertRows<ExpertRows<P>> { static constexpr bool value = true, pairs = P; };

template <int BM, int BN, int WGM, int WGN, int STAGES, typename TOut, int SW = 0, typename GS = GroupStride>
__global__ __launch_bounds__(64 * WGM * WGN) void gemm_dl_tile_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                      const void* __restrict__ bias, int bias_f32,
                                                                      TOut* __restrict__ out, int M, int N, int K, int ldx, int ldo,
                                                                      int out_cols, int k_per_split, GS gs) {
    constexpr bool EX = IsExpertRows<GS>::value;
    static_assert(!EX || (!SW && sizeof(TOut) == 2), "groups of rows: bfloat16 results with an activation of their own");
    static_assert(!SW || (BN / WGN) % 64 == 0, "the fused gate needs whole 64-row blocks per wave");
    // A slab row holds PPR pieces of 16 bytes; one load instruction of a wave fills RPL rows.
    constexpr int TK = 64, PPR = TK / 8, RPL = 64 / PPR;
    // Split K (k_per_split > 0, a multiple of 64): blockIdx.y owns the columns [y * k_per_split, ...) of
    // x and w and writes its own [M, ldo] slab of partial sums to out; whoever reads them adds the slabs up.
    const int ldw = K;
    if constexpr (!EX) {
        x += blockIdx.z * gs.x;
        w += blockIdx.z * gs.w;
        out += blockIdx.z * gs.out;
        if (k_per_split > 0) {
            const int kb = blockIdx.y * k_per_split;
            x += kb;
            w += kb;
            out += (size_t)blockIdx.y * M * ldo;
            K = min(K - kb, k_per_split);
        }
    }
    constexpr int NW = WGM * WGN;
    constexpr int WM = BM / WGM, WN = BN / WGN;          // wave tile
    constexpr int FM = WM / 16, FN = WN / 16;            // 16x16 blocks per wave
    constexpr int ROWS = BM + BN;
    constexpr int LROWS = dl_slab_rows(BM, BN, NW);  // a slab's rows in shared memory: ROWS, rounded up so that ...
    constexpr int LOADS = LROWS / RPL / NW;              // ... every wave issues as many load instructions per slab (RPL rows each)
    static_assert(LOADS * (STAGES - 1) < 64, "outstanding loads must fit the counter");
    extern __shared__ __attribute__((aligned(16))) bf16_t lds_raw[];   // [STAGES][LROWS][TK]

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WGN, wn = wave % WGN;
    // tile order as in gemm_mfma_tile_kernel: each XCD walks 8 x 8 blocks of tiles out of its own L2
    const int tiles_n = (N + BN - 1) / BN;
    int m0, n0, m_base = 0;                                 // (m_base: the row that the lanes' offsets into x count from)
    if constexpr (EX) {
        int first = 0, at = -1, count = 0, lo = 0, total = 0, lid = 0;
        for (int pass = gs.groups > TL_WAVE ? 0 : 1; pass < 2; ++pass) {      // more groups than lanes: the tiles are counted first
            first = 0;
            for (int base = 0; base < gs.groups && at < 0; base += TL_WAVE) {
                const int e = base + lane;
                const int from = e < gs.groups ? gs.offsets[e] : 0;
                const int mine = e < gs.groups ? (gs.offsets[e + 1] - from + BM - 1) / BM : 0;
                int upto = mine;
#pragma unroll
                for (int o = 1; o < TL_WAVE; o <<= 1) {
                    const int t = __shfl_up(upto, o, TL_WAVE);
                    if (lane >= o) upto += t;
                }
                const int sum = __builtin_amdgcn_readlane(upto, TL_WAVE - 1);
                if (pass == 1) {
                    if (gs.groups <= TL_WAVE) total = sum;
                    const int all = total * tiles_n;
                    if ((int)blockIdx.x >= all) return;
                    const int xcd = blockIdx.x % 8, idx = blockIdx.x / 8;
                    lid = xcd * (all / 8) + min(xcd, all % 8) + idx;
                    const unsigned long long past = __ballot((first + upto) * tiles_n > lid);
                    if (past) {
                        const int l = __builtin_amdgcn_readfirstlane(__ffsll(past) - 1);
                        at = base + l;
                        count = __builtin_amdgcn_readlane(mine, l);
                        lo = __builtin_amdgcn_readlane(from, l);
                        first += __builtin_amdgcn_readlane(upto, l) - count;
                        break;
                    }
                }
                first += sum;
            }
            if (pass == 0) total = first;
        }
        const int local = lid - first * tiles_n;
        m0 = lo + (local % count) * BM;
        n0 = (local / count) * BN;
        M = gs.offsets[at + 1];
        w += (size_t)at * N * K;
    } else {
        const int tiles_m = (M + BM - 1) / BM;
        int lid;
        {
            const int total = gridDim.x, xcd = blockIdx.x % 8, idx = blockIdx.x / 8;
            lid = xcd * (total / 8) + min(xcd, total % 8) + idx;
        }
        const int per_group = 8 * tiles_n;
        const int first_m = (lid / per_group) * 8;
        const int rows = min(tiles_m - first_m, 8);
        m0 = (first_m + (lid % per_group) % rows) * BM;
        n0 = ((lid % per_group) / rows) * BN;
        m_base = m0;
    }

    // Instruction j of this wave fills rows RPL (wave + j NW) .. + RPL of the stacked [x rows; w rows] slab.  Its
    // eight rows are all of x or all of w (BM is a multiple of RPL), so its address is a base the wave shares (the
    // tile's first row of x or of w, moved along K from step to step by scalar instructions) and a 32-bit offset per
    // lane that never changes: half the address registers of a 64-bit address per lane, and no vector addition per
    // request (2048 x 37888 x 3584: 500 -> 478 us).
    static_assert(BM % RPL == 0, "the rows of one request lie in one operand");
    int ldst[LOADS];
    unsigned soff[LOADS];
    unsigned of_x = 0;                                      // bit j: request j fetches rows of x
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
        const int base_row = RPL * (wave + j * NW);
        const int row = min(base_row + lane / PPR, ROWS - 1);      // (rows of the rounding: copies of the last row, never read)
        const int c = (lane % PPR) ^ ((row >> 1) & 7);
        if (row < BM) {
            int m = min(m0 + row, M - 1);
            if constexpr (EX) m = gs.src ? gs.src[m] : m;
            soff[j] = (unsigned)((m - m_base) * ldx + c * 8) * 2;
        }
        else soff[j] = (unsigned)((min(n0 + row - BM, N - 1) - n0) * ldw + c * 8) * 2;
        ldst[j] = __builtin_amdgcn_readfirstlane(base_row * TK * 2);
        of_x |= (unsigned)(base_row < BM) << j;
    }
    of_x = __builtin_amdgcn_readfirstlane(of_x);
    const bf16_t* xt = x + (size_t)m_base * ldx;
    const bf16_t* wt = w + (size_t)n0 * ldw;
    const unsigned lds_base = (unsigned)(uintptr_t)((void __attribute__((address_space(3)))*)lds_raw);

    f32x4_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[i][j][v] = 0.f;

    // Products of 16 x 16 x 32: lane l holds eight columns of K, 8 (l / 16) .. + 7 of a phase's 32, of row l % 16 of a block.  They do the work of a 32 x 32 x
    // 16 product in as many cycles and move half as much of the accumulators, and the power that this takes is what sets the clock of a large product (2650 cycles a slab at
    // 1.67 GHz with the larger blocks, 2610 at 1.8 with these; with all that follows 8192 x 8192 x 8192 850 -> 766 us, 2048 x 37888 x 3584 475 -> 431, 2048 x 8192 x 2048 62 -> 54).
    //
    // The loop is a hand-laid pipeline; scheduling fences keep the compiler from undoing it.  A step of TK columns has two phases of FM * FN products.  A phase's
    // memory instructions go between its products, one product first: the operand reads of the next phase, so that a read has a whole phase to arrive.  (All
    // reads first and then all products, the wait at the loop's head came out as one for every read, the ones just issued too.)  Both operands
    // have two sets of registers; where these and the sums do not fit (the waves of 64 x 160), the operand with more blocks (`rolled`) has one set, each
    // block read anew once the last product that needs it is under way (in a wave of 128 x 64, where both ways fit, it costs a fortieth).
    //
    // The last phase of a step waits for the next slab and meets the other waves at the barrier (they have all read their last operands of this
    // slab by then): at its start, or with many products three quarters through it, which leaves the slab that much longer to arrive (8192 x 8192 x 8192: 863 us at the
    // start, 780 halfway, 775 at three quarters; 766 with two memory instructions behind a product).  Behind the barrier go the first half of the requests for the slab STAGES - 1 ahead, into
    // the buffer just given up, and the reads of the first operands of the next slab.  The other half of the requests goes into the first phase of the next
    // step: a compute unit's 64 requests in one phase hold its waves up, whatever they fetch (requests of 4 bytes a lane cost the same; without any the loop ran a
    // sixth faster), and in two phases less so (all of them behind the reads: 857 us).  Past the end the last slab is requested again (nobody reads it), so the count
    // of requests in flight is the same in every step, which the wait relies on.
    constexpr int PHASES = TK / 32, NM = FM * FN;
    constexpr bool MANY = NM > 16, ROLL_X = FM >= FN;
    constexpr bool ROLL = 4 * NM + 8 * (FM + FN) > (NW > 4 ? 232 : 464);      // registers of the products and of two sets of operands
    constexpr int FR = ROLL_X ? FM : FN, FD = ROLL_X ? FN : FM;       // blocks of the rolled operand (the outer index of the products) and of the other
    constexpr int BARRIER_AT = MANY ? NM * 3 / 4 : 0;                    // products of the last phase ahead of its barrier
    Frag16 rolled[ROLL ? 1 : 2][FR], paired[2][FD];
    const int slabs = K / TK;
    const int fr = lane & 15, fq = lane >> 4;
    // where this lane's first block lies in a slab (rows are 64 elements; a block's rows are 1024 further on, its slots' order the same)
    const int x_at = (wm * WM + fr) * TK, w_at = (BM + wn * WN + fr) * TK;
    const int roll_at = ROLL_X ? x_at : w_at, pair_at = ROLL_X ? w_at : x_at;
    const int slot[PHASES] = {(fq ^ ((fr >> 1) & 7)) * 8, ((fq + 4) ^ ((fr >> 1) & 7)) * 8};
    // requests of a slab issued in the last phase of a step; the rest in the next step's first.  (Not for the smallest tile,
    // four requests a wave and slab: split in two they made the decode step's products over K a fiftieth slower.)
    constexpr int L_LAST = LOADS >= 6 ? (LOADS + 1) / 2 : LOADS;
    auto request = [&](int slab, int j) {
        // (which operand request j fetches is known at compile time where the waves' requests cover whole multiples of x's rows)
        const bool from_x = BM % (RPL * NW) == 0 ? j < BM / (RPL * NW) : (bool)((of_x >> j) & 1);
        const bf16_t* from = (from_x ? xt : wt) + min(slab, slabs - 1) * TK;
        load_to_lds_at(from, soff[j], lds_base + (slab % STAGES) * LROWS * TK * 2 + ldst[j]);
    };
#pragma unroll
    for (int st = 0; st < STAGES - 1; ++st)
#pragma unroll
        for (int j = 0; j < LOADS; ++j) request(st, j);
    wait_direct_loads<(STAGES - 2) * LOADS>();
    __syncthreads();
#pragma unroll
    for (int j = 0; j < L_LAST; ++j) request(STAGES - 1, j);
#pragma unroll
    for (int d = 0; d < FD; ++d) paired[0][d].u = *(const uint4*)(lds_raw + pair_at + d * 16 * TK + slot[0]);
#pragma unroll
    for (int r = 0; r < FR; ++r) rolled[0][r].u = *(const uint4*)(lds_raw + roll_at + r * 16 * TK + slot[0]);
    __builtin_amdgcn_sched_barrier(0);

    for (int sl = 0; sl < slabs; ++sl) {
#pragma unroll
        for (int kk = 0; kk < PHASES; ++kk) {
            const int cur = kk & 1, nxt = cur ^ 1;
            const bool last = kk + 1 == PHASES;
            const bf16_t* nb = lds_raw + ((sl + (last ? 1 : 0)) % STAGES) * LROWS * TK + slot[last ? 0 : kk + 1];      // where the next phase's operands lie
            // this phase's requests [lfirst, lend) and the slab they fetch: in the last phase the slab that gets the
            // buffer given up now, in the first the rest of the slab that got the buffer given up a step ago
            const int lfirst = last ? 0 : L_LAST, lend = last ? L_LAST : kk == 0 ? LOADS : L_LAST;
            const int slab_of = last ? sl + STAGES : sl - 1 + STAGES;
            const int nl = lend - lfirst;
            const int start = last ? BARRIER_AT : 0;                                         // the first product that memory instructions follow
            const int ops = nl + FD + FR;                                                    // memory instructions of this phase ...
            const int least = (ops + NM - start - 1) / (NM - start), per = MANY && !ROLL && least < 2 ? 2 : least;      // ... and how many follow each product
            auto issue = [&](int op) {
                if (op < nl) request(slab_of, lfirst + op);
                else if (op < nl + FD) paired[nxt][op - nl].u = *(const uint4*)(nb + pair_at + (op - nl) * 16 * TK);
                else rolled[ROLL ? 0 : nxt][op - nl - FD].u = *(const uint4*)(nb + roll_at + (op - nl - FD) * 16 * TK);
            };
            int op = 0;
#pragma unroll
            for (int q = 0; q < NM; ++q) {
                if (last && q == start) {
                    wait_direct_loads<(STAGES - 2) * LOADS>();
                    __syncthreads();
                    __builtin_amdgcn_sched_barrier(0);
                }
                const int r = q / FD, d = q % FD, i = ROLL_X ? r : d, j = ROLL_X ? d : r;
                const Frag16 &fx = ROLL_X ? rolled[ROLL ? 0 : cur][r] : paired[cur][d], &fw = ROLL_X ? paired[cur][d] : rolled[ROLL ? 0 : cur][r];
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw.v, fx.v, acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (q < start) continue;
#pragma unroll
                for (int e = 0; e < per; ++e) {
                    if (op >= ops || (ROLL && op >= nl + FD && q < (op - nl - FD + 1) * FD - 1)) break;      // (a rolled block that products to come still need stays)
                    issue(op++);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (; op < ops; ++op) issue(op);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    wait_direct_loads<0>();

    // The products are taken as weight block times x block, so of a 16x16 block a lane holds one row of x, m = lane % 16, and four neighbouring
    // output columns, 4 (lane / 16) and up.  With the fused gate, of every four blocks of columns the first two hold gate columns and the
    // other two the up columns of the same 32 outputs.
    const int lm = lane & 15, quad = lane >> 4;
    if constexpr (EX) {
        store_expert_tile<BM, BN, WM, WN, FM, FN, STAGES * ROWS * TK, IsExpertRows<GS>::pairs>(acc, lds_raw + wave * (WM * (IsExpertRows<GS>::pairs ? WN / 2 : WN)),
            out, m0 + wm * WM, n0 + wn * WN, M, N, ldo, gs.act);
        return;
    }
    constexpr int WNO = SW ? WN / 2 : WN;                   // output columns of a wave tile
    constexpr int FNO = SW ? FN / 2 : FN;                   // and its blocks of 16 of them
    const int cols = SW ? out_cols : N;                     // output columns in all
    const int c0 = (SW ? n0 / 2 : n0) + wn * WNO;           // first output column and row of this wave
    const int r0 = m0 + wm * WM;
    auto value = [&](int i, int jo, int v) -> float {
        if constexpr (SW) return gate_mul<SW>(acc[i][jo / 2 * 4 + jo % 2][v], acc[i][jo / 2 * 4 + 2 + jo % 2][v]);
        else return acc[i][jo][v];
    };
    auto bias_at = [&](int n) -> float { return (!SW && bias && n < cols) ? load_vec(bias, bias_f32, n) : 0.f; };

    if constexpr (sizeof(TOut) == 2) {
        if (cols % 8 == 0 && ldo % 8 == 0 && ((uintptr_t)out % 16) == 0) {
            // bfloat16 rows that can be stored in 16-byte pieces: the wave lays its tile out row by
            // row in shared memory (the slab buffers are free now; 16-byte piece c of row r in slot
            // c ^ (r % CX) against bank conflicts) and stores it in whole rows, 64 lanes times 16
            // bytes per instruction, instead of two bytes per lane and store.
            constexpr int C = WNO / 8;
            constexpr int CX = C & -C;                       // the slots are exchanged within groups of CX, a power of two
            static_assert((WM * C) % 64 == 0, "the rows of a wave tile must divide over its lanes");
            static_assert(BM * (SW ? BN / 2 : BN) <= STAGES * ROWS * TK, "the result tile must fit the slab buffers");
            __syncthreads();
            bf16_t* stage = lds_raw + wave * (WM * WNO);
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int jo = 0; jo < FNO; ++jo) {
                    const int n = jo * 16 + 4 * quad, row = i * 16 + lm;
                    bf16_t h[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) h[e] = from_float<bf16_t>(value(i, jo, e) + bias_at(c0 + n + e));
                    uint2 packed;
                    packed.x = (uint32_t)h[0].bits | ((uint32_t)h[1].bits << 16);
                    packed.y = (uint32_t)h[2].bits | ((uint32_t)h[3].bits << 16);
                    *(uint2*)(stage + row * WNO + (((n >> 3) ^ (row & (CX - 1))) * 8) + (n & 4)) = packed;
                }
            // (one wave's shared-memory accesses are carried out in order: no wait in between)
#pragma unroll
            for (int q = 0; q < WM * C / 64; ++q) {
                const int idx = q * 64 + lane;
                const int row = idx / C, piece = idx % C;
                const uint4 val = *(const uint4*)(stage + row * WNO + ((piece ^ (row & (CX - 1))) * 8));
                const int m = r0 + row, n = c0 + piece * 8;
                if (m < M && n < cols) *(uint4*)((bf16_t*)out + (size_t)m * ldo + n) = val;
            }
            return;
        }
    }
    const bool quads = sizeof(TOut) == 4 && cols % 4 == 0 && ldo % 4 == 0 && ((uintptr_t)out % 16) == 0;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int m = r0 + i * 16 + lm;
        if (m >= M) continue;
#pragma unroll
        for (int jo = 0; jo < FNO; ++jo) {
            const int n = c0 + jo * 16 + 4 * quad;
            if (quads) {
                if (n < cols) {
                    float4 f;
                    f.x = value(i, jo, 0) + bias_at(n);
                    f.y = value(i, jo, 1) + bias_at(n + 1);
                    f.z = value(i, jo, 2) + bias_at(n + 2);
                    f.w = value(i, jo, 3) + bias_at(n + 3);
                    *(float4*)((float*)out + (size_t)m * ldo + n) = f;
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < cols) out[(size_t)m * ldo + n + e] = from_float<TOut>(value(i, jo, e) + bias_at(n + e));
            }
        }
    }
}
