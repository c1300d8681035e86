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
constexpr int dl_slab_rows(int bm, int bn, int waves, int tk) {
    const int per = (64 / (tk / 8)) * waves;
    return (bm + bn + per - 1) / per * per;
}

// The result tile of a group of rows: the activation applied to the accumulators (PAIRS: to a lane's neighbouring columns 2i and 2i + 1, which give
// one output column), laid out row by row in the free slab buffers as below and stored in whole rows.
template <int ACT>
__device__ __forceinline__ float activated(float v) { return activate(v, ACT); }

template <int ACT, int BM, int BN, int WM, int WN, int FM, int FN, int ROOM, bool PAIRS>
__device__ __forceinline__ void store_expert_tile_as(const f32x16_t (&acc)[FM][FN], bf16_t* stage, bf16_t* out, int r0, int c0, int M, int N, int ldo) {
    constexpr int WNO = PAIRS ? WN / 2 : WN;
    static_assert(BM * (PAIRS ? BN / 2 : BN) <= ROOM, "the result tile must fit the slab buffers");
    const int lane = threadIdx.x & 63, lm = lane & 31, half = lane >> 5;
    const int cols = PAIRS ? N / 2 : N, co = PAIRS ? c0 / 2 : c0;
    const bool whole = cols % 8 == 0 && ldo % 8 == 0 && ((uintptr_t)out % 16) == 0;
    constexpr int C = WNO / 8, CX = C & -C;
    static_assert((WM * C) % 64 == 0, "the rows of a wave tile must divide over its lanes");
    if (whole) __syncthreads();
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                constexpr int V = PAIRS ? 2 : 4;              // output columns of a lane's four
                bf16_t h[V];
#pragma unroll
                for (int e = 0; e < V; ++e) {
                    if constexpr (PAIRS) h[e] = from_float<bf16_t>(activated<ACT>(acc[i][j][4 * g + 2 * e]) * acc[i][j][4 * g + 2 * e + 1]);
                    else h[e] = from_float<bf16_t>(activated<ACT>(acc[i][j][4 * g + e]));
                }
                const int n = (j * 32 + 8 * g + 4 * half) / (PAIRS ? 2 : 1), row = i * 32 + lm;
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
__device__ __forceinline__ void store_expert_tile(const f32x16_t (&acc)[FM][FN], bf16_t* stage, bf16_t* out, int r0, int c0, int M, int N, int ldo, int act) {
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

template <int BM, int BN, int WGM, int WGN, int STAGES, typename TOut, int SW = 0, int TK = 64, typename GS = GroupStride>
__global__ __launch_bounds__(64 * WGM * WGN) void gemm_dl_tile_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                      const void* __restrict__ bias, int bias_f32,
                                                                      TOut* __restrict__ out, int M, int N, int K, int ldx, int ldo,
                                                                      int out_cols, int k_per_split, GS gs) {
    constexpr bool EX = IsExpertRows<GS>::value;
    static_assert(!EX || (!SW && sizeof(TOut) == 2), "groups of rows: bfloat16 results with an activation of their own");
    static_assert(!SW || (BN / WGN) % 64 == 0, "the fused gate needs whole 64-row blocks per wave");
    static_assert(TK == 64 || TK == 32, "slabs of 64 or 32 columns");
    // A slab row holds PPR pieces of 16 bytes; one load instruction of a wave fills RPL rows.  With
    // slabs of 32 columns a row is 64 bytes and piece c of row r lies in slot c ^ ((r >> 2) & 3): the
    // sixteen rows a quarter-wave reads then fall on all 64 banks as well.  Half the slab is half the
    // shared memory per stage: twice as many stages fit, and a request has twice as long to arrive.
    constexpr int PPR = TK / 8, RPL = 64 / PPR;
#define DL_SWZ(r) (TK == 64 ? (((r) >> 1) & 7) : (((r) >> 2) & 3))
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
    constexpr int FM = WM / 32, FN = WN / 32;            // 32x32 blocks per wave
    constexpr int ROWS = BM + BN;
    constexpr int LROWS = dl_slab_rows(BM, BN, NW, TK);  // a slab's rows in shared memory: ROWS, rounded up so that ...
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
        const int c = (lane % PPR) ^ DL_SWZ(row);
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

    f32x16_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    const int slabs = K / TK;
    const int fr = lane & 31, fh = lane >> 5;
    int arow[FM], brow[FN], akey[FM], bkey[FN];
#pragma unroll
    for (int i = 0; i < FM; ++i) { arow[i] = wm * WM + i * 32 + fr; akey[i] = DL_SWZ(arow[i]); }
#pragma unroll
    for (int j = 0; j < FN; ++j) { brow[j] = BM + wn * WN + j * 32 + fr; bkey[j] = DL_SWZ(brow[j]); }
#undef DL_SWZ

    // The loop is a hand-laid pipeline; scheduling fences keep the compiler from undoing it.  A step
    // of TK columns has TK / 16 phases of FM * FN products.  A phase's memory instructions go between
    // its products, one product first: the operand reads of the next phase into the other register set,
    // so a read has a whole phase to arrive, and the wait before a phase's first product is for operands
    // asked for a phase ago with nothing younger outstanding.  (All reads first and then all products,
    // the wait at the loop's head came out as one for every read, the ones just issued too, and the 7B's fused
    // gate/up product at 2048 rows took 537 us instead of 487.)  The last phase of a step first waits for the
    // next slab and meets the other waves at the barrier (they have all read their last operands of this
    // slab by then); between its products go the first half of the requests for the slab STAGES - 1 ahead, into
    // the buffer just given up, and then the reads of the first operands of the next slab.  The other half of
    // the requests goes into the first phase of the next step: a compute unit's 64 requests in one phase hold
    // its waves up, whatever they fetch (requests of 4 bytes a lane cost the same; without any the loop ran a
    // sixth faster), and in two phases less so (2048 x 3584 x 18944: 392 -> 353 us; spread over three phases the
    // last ones arrive too late).  Past the end the last slab is requested again (nobody reads it), so the count
    // of requests in flight is the same in every step, which the wait relies on.
    Frag16 af[2][FM], bfr[2][FN];
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
    for (int i = 0; i < FM; ++i) af[0][i].u = *(const uint4*)(lds_raw + arow[i] * TK + ((fh ^ akey[i]) * 8));
#pragma unroll
    for (int j = 0; j < FN; ++j) bfr[0][j].u = *(const uint4*)(lds_raw + brow[j] * TK + ((fh ^ bkey[j]) * 8));
    __builtin_amdgcn_sched_barrier(0);

    constexpr int PHASES = TK / 16;
    constexpr int NM = FM * FN, NR = FM + FN;               // products and operand reads of a phase
    for (int sl = 0; sl < slabs; ++sl) {
        const bf16_t* cb = lds_raw + (sl % STAGES) * LROWS * TK;
#pragma unroll
        for (int kk = 0; kk < PHASES; ++kk) {
            const int cur = kk & 1, nxt = cur ^ 1;
            const bool last = kk + 1 == PHASES;
            const bf16_t* nb = last ? lds_raw + ((sl + 1) % STAGES) * LROWS * TK : cb;      // where the next phase's operands lie
            const int c = (last ? 0 : 2 * (kk + 1)) + fh;
            // this phase's requests [lfirst, lend) and the slab they fetch: in the last phase the slab that gets the
            // buffer given up now, in the first the rest of the slab that got the buffer given up a step ago
            const int lfirst = last ? 0 : L_LAST, lend = last ? L_LAST : kk == 0 ? LOADS : L_LAST;
            const int slab_of = last ? sl + STAGES : sl - 1 + STAGES;
            const int nl = lend - lfirst;
            const int ops = nl + NR;                                                         // memory instructions of this phase ...
            const int per = (ops + NM - 1) / NM;                                             // ... and how many follow each product
            if (last) {
                wait_direct_loads<(STAGES - 2) * LOADS>();
                __syncthreads();
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (NM == 1) {
                // One product a phase (the smallest tile): a phase's memory instructions first, then its product, which
                // covers them; but for the step's first phase, whose product comes first so that the wait at the loop's
                // head is for that product's operands alone.
                if (kk == 0) {
                    acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[cur][0].v, af[cur][0].v, acc[0][0], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int op = 0; op < ops; ++op) {
                    const int r = op - nl;
                    if (r < 0) request(slab_of, lfirst + op);
                    else if (r < FM) af[nxt][r].u = *(const uint4*)(nb + arow[r] * TK + ((c ^ akey[r]) * 8));
                    else bfr[nxt][r - FM].u = *(const uint4*)(nb + brow[r - FM] * TK + ((c ^ bkey[r - FM]) * 8));
                }
                __builtin_amdgcn_sched_barrier(0);
                if (kk > 0) {
                    acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[cur][0].v, af[cur][0].v, acc[0][0], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
                continue;
            }
            int op = 0;
#pragma unroll
            for (int q = 0; q < NM; ++q) {
                acc[q / FN][q % FN] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[cur][q % FN].v, af[cur][q / FN].v, acc[q / FN][q % FN], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int e = 0; e < per; ++e, ++op) {
                    if (op >= ops) break;
                    const int r = op - nl;
                    if (r < 0) request(slab_of, lfirst + op);
                    else if (r < FM) af[nxt][r].u = *(const uint4*)(nb + arow[r] * TK + ((c ^ akey[r]) * 8));
                    else bfr[nxt][r - FM].u = *(const uint4*)(nb + brow[r - FM] * TK + ((c ^ bkey[r - FM]) * 8));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    wait_direct_loads<0>();

    // The products are taken as weight block times x block, so of a 32x32 block a lane holds one
    // row of x, m = lane % 32, and sixteen output columns n = 8 (v / 4) + 4 (lane / 32) + v % 4:
    // four neighbours at a time.  With the fused gate, even blocks hold gate columns and the next
    // block the up columns of the same 32 outputs.
    const int lm = lane & 31, half = lane >> 5;
    if constexpr (EX) {
        store_expert_tile<BM, BN, WM, WN, FM, FN, STAGES * ROWS * TK, IsExpertRows<GS>::pairs>(acc, lds_raw + wave * (WM * (IsExpertRows<GS>::pairs ? WN / 2 : WN)),
            out, m0 + wm * WM, n0 + wn * WN, M, N, ldo, gs.act);
        return;
    }
    constexpr int WNO = SW ? WN / 2 : WN;                   // output columns of a wave tile
    constexpr int FNO = SW ? FN / 2 : FN;                   // and its blocks of 32 of them
    const int cols = SW ? out_cols : N;                     // output columns in all
    const int c0 = (SW ? n0 / 2 : n0) + wn * WNO;           // first output column and row of this wave
    const int r0 = m0 + wm * WM;
    auto value = [&](int i, int jo, int v) -> float {
        if constexpr (SW) return gate_mul<SW>(acc[i][2 * jo][v], acc[i][2 * jo + 1][v]);
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
                for (int jo = 0; jo < FNO; ++jo)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const int n = jo * 32 + 8 * g + 4 * half;
                        bf16_t h[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) h[e] = from_float<bf16_t>(value(i, jo, 4 * g + e) + bias_at(c0 + n + e));
                        uint2 packed;
                        packed.x = (uint32_t)h[0].bits | ((uint32_t)h[1].bits << 16);
                        packed.y = (uint32_t)h[2].bits | ((uint32_t)h[3].bits << 16);
                        const int row = i * 32 + lm;
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
        const int m = r0 + i * 32 + lm;
        if (m >= M) continue;
#pragma unroll
        for (int jo = 0; jo < FNO; ++jo)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int n = c0 + jo * 32 + 8 * g + 4 * half;
                if (quads) {
                    if (n < cols) {
                        float4 f;
                        f.x = value(i, jo, 4 * g) + bias_at(n);
                        f.y = value(i, jo, 4 * g + 1) + bias_at(n + 1);
                        f.z = value(i, jo, 4 * g + 2) + bias_at(n + 2);
                        f.w = value(i, jo, 4 * g + 3) + bias_at(n + 3);
                        *(float4*)((float*)out + (size_t)m * ldo + n) = f;
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (n + e < cols) out[(size_t)m * ldo + n + e] = from_float<TOut>(value(i, jo, 4 * g + e) + bias_at(n + e));
                }
            }
    }
}

