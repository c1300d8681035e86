// Matrix products over groups (one weight matrix per group: an expert and the tokens routed to it, or a head and
// its slice of every token's row), the router's choice of experts, the sort of tokens by expert, the weighted sum
// of the chosen experts' outputs, and the elementwise activation of a dense feed-forward.  Sums are float.
#include "row_ring.h"

// ------------------------------------------------------------------ grouped product
// out[row(m), g_out + n] = act(sum_k a[src(m), g_a + k] * w[g][n][k]) for the rows m of group g, in tiles of 64 x 64
// with K in steps of 16 through shared memory; a thread owns a 4 x 4 block of the tile.  One order of summation per
// output element whatever else is in the step.
//   offsets == null: every group has the same `rows` rows (row m is token m), group g reads the columns from
//                    g * a_group on and writes the columns from g * out_group on; blockIdx.z is the group.
//   offsets != null: group g owns the rows offsets[g] .. offsets[g + 1] - 1 (sorted slots); blockIdx.x runs over an upper
//                    bound of all groups' tiles and finds its group by walking the offsets; `src` (optional) maps a
//                    sorted slot to the row of `a` it reads (a token routed to an expert), output rows are the slots.
//   gate (optional, without offsets, no activation): out[m, c] is multiplied by sigmoid(gate[m, c]) before its one rounding (row m of `gate`
//                    is gate_ld numbers after the one before, of the activation type).
#define GG_T 64
#define GG_K 16

template <typename T>
__global__ void __launch_bounds__(256)
grouped_gemm_kernel(const T* __restrict__ a, int a_ld, int a_group, const int* __restrict__ src, const T* __restrict__ w,
                    T* __restrict__ out, int out_ld, int out_group, const int* __restrict__ offsets, int groups, int rows,
                    int N, int K, int act, const T* __restrict__ gate, int gate_ld) {
    __shared__ float sa[GG_K][GG_T + 4];
    __shared__ float sw[GG_K][GG_T + 4];
    int g, m0, m_end;
    if (offsets == nullptr) {
        g = blockIdx.z; m0 = blockIdx.x * GG_T; m_end = rows;
        if (m0 >= m_end) return;
    } else {
        int tile = blockIdx.x;
        g = 0; m0 = -1; m_end = 0;
        for (int e = 0; e < groups; ++e) {
            const int lo = offsets[e], hi = offsets[e + 1], tiles = (hi - lo + GG_T - 1) / GG_T;
            if (tile < tiles) { g = e; m0 = lo + tile * GG_T; m_end = hi; break; }
            tile -= tiles;
        }
        if (m0 < 0) return;
    }
    const int n0 = blockIdx.y * GG_T;
    const T* wg = w + (size_t)g * N * K;
    const int a_col = offsets == nullptr ? g * a_group : 0, out_col = offsets == nullptr ? g * out_group : 0;
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;      // the thread's block: rows ty*4.., columns tx*4..
    // loads: a thread fetches 4 elements of a and 4 of w per step: row lr of the tile, k = lk .. lk+3
    const int lr = threadIdx.x / 4, lk = (threadIdx.x % 4) * 4;
    const int am = m0 + lr;
    const T* arow = nullptr;
    if (am < m_end) arow = a + (size_t)(src ? src[am] : am) * a_ld + a_col;
    const T* wrow = (n0 + lr < N) ? wg + (size_t)(n0 + lr) * K : nullptr;
    float acc[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += GG_K) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = k0 + lk + u;
            sa[lk + u][lr] = (arow && k < K) ? to_float(arow[k]) : 0.f;
            sw[lk + u][lr] = (wrow && k < K) ? to_float(wrow[k]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < GG_K; ++k) {
            float av[4], wv[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) { av[u] = sa[k][ty * 4 + u]; wv[u] = sw[k][tx * 4 + u]; }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(av[i], wv[j], acc[i][j]);
        }
        __syncthreads();
    }
    const int base_act = act & ~ACT_PAIRS;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + ty * 4 + i;
        if (m >= m_end) continue;
        T* orow = out + (size_t)m * out_ld + out_col;
        if (act & ACT_PAIRS) {                          // (N is even: a pair lies in one thread's four columns)
#pragma unroll
            for (int j = 0; j < 4; j += 2) {
                const int n = n0 + tx * 4 + j;
                if (n + 1 < N) orow[n / 2] = from_float<T>(activate(acc[i][j], base_act) * acc[i][j + 1]);
            }
            continue;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + tx * 4 + j;
            if (n >= N) continue;
            float v = activate(acc[i][j], act);
            if (gate) v *= sigmoid(to_float(gate[(size_t)m * gate_ld + out_col + n]));
            orow[n] = from_float<T>(v);
        }
    }
}

// The same product on the matrix cores (bfloat16, K a multiple of 32, 16-byte aligned rows): both operands have K side by
// side in memory, which is how v_mfma_f32_16x16x32_bf16 wants them, so a lane fetches its 16-byte pieces straight from
// memory (the weights' once per tile of rows, the rows' from the caches) and nothing passes through shared memory.  The
// weights are the first operand, so that a lane ends up with four neighbouring output columns of one row.  A work-group
// of four waves owns a tile of 32 rows x 256 columns (one wave: 32 x 64); few rows per group (a decode step's experts)
// leave half of each product empty, which costs nothing where the weights' stream sets the time.
#define GM_BM 32
#define GM_BN 256

typedef __bf16 gm_bf16x8 __attribute__((ext_vector_type(8)));
typedef float gm_f32x4 __attribute__((ext_vector_type(4)));
union GmFrag {
    uint4 u;
    gm_bf16x8 v;
};

__global__ void __launch_bounds__(256)
grouped_gemm_mfma_kernel(const bf16_t* __restrict__ a, int a_ld, int a_group, const int* __restrict__ src, const bf16_t* __restrict__ w,
                         bf16_t* __restrict__ out, int out_ld, int out_group, const int* __restrict__ offsets, int groups, int rows,
                         int N, int K, int act, const bf16_t* __restrict__ gate, int gate_ld) {
    int g, m0, m_end;
    if (offsets == nullptr) {
        g = blockIdx.z; m0 = blockIdx.x * GM_BM; m_end = rows;
        if (m0 >= m_end) return;
    } else {
        int tile = blockIdx.x;
        g = 0; m0 = -1; m_end = 0;
        for (int e = 0; e < groups; ++e) {
            const int lo = offsets[e], hi = offsets[e + 1], tiles = (hi - lo + GM_BM - 1) / GM_BM;
            if (tile < tiles) { g = e; m0 = lo + tile * GM_BM; m_end = hi; break; }
            tile -= tiles;
        }
        if (m0 < 0) return;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, kg = lane >> 4;
    const int n0 = blockIdx.y * GM_BN + wave * 64;
    if (n0 >= N) return;
    const bf16_t* wg = w + (size_t)g * N * K;
    const int a_col = offsets == nullptr ? g * a_group : 0, out_col = offsets == nullptr ? g * out_group : 0;
    // this lane's rows of the two operands: weight row n0 + 16 i + li (clamped), x row of tile row 16 j + li (clamped)
    const bf16_t* wrow[4];
    const bf16_t* xrow[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) wrow[i] = wg + (size_t)min(n0 + 16 * i + li, N - 1) * K + 8 * kg;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int m = min(m0 + 16 * j + li, m_end - 1);
        xrow[j] = a + (size_t)(src ? src[m] : m) * a_ld + a_col + 8 * kg;
    }
    const bool second = m0 + 16 < m_end;                // the tile has rows beyond its first 16
    gm_f32x4 acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = gm_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int k = 0; k < K; k += 32) {
        GmFrag wf[4], xf[2];
#pragma unroll
        for (int i = 0; i < 4; ++i) wf[i].u = *(const uint4*)(wrow[i] + k);
        xf[0].u = *(const uint4*)(xrow[0] + k);
        if (second) xf[1].u = *(const uint4*)(xrow[1] + k);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i].v, xf[0].v, acc[i][0], 0, 0, 0);
            if (second) acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i].v, xf[1].v, acc[i][1], 0, 0, 0);
        }
    }
    // acc[i][j][v] = out[row 16 j + li][column n0 + 16 i + 4 kg + v]
    const int base_act = act & ~ACT_PAIRS;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int m = m0 + 16 * j + li;
        if (m >= m_end) continue;
        bf16_t* orow = out + (size_t)m * out_ld + out_col;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n = n0 + 16 * i + 4 * kg;
            if (act & ACT_PAIRS) {                      // a lane's four columns are two pairs: two outputs at column n / 2
#pragma unroll
                for (int v = 0; v < 4; v += 2)
                    if (n + v + 1 < N) orow[(n + v) / 2] = from_float<bf16_t>(activate(acc[i][j][v], base_act) * acc[i][j][v + 1]);
                continue;
            }
            if (gate) {                                 // (no activation beside a gate)
                const bf16_t* grow = gate + (size_t)m * gate_ld + out_col;
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[i][j][v] *= sigmoid(to_float(grow[min(n + v, N - 1)]));
            }
            if (n + 3 < N && ((out_ld | out_col) & 3) == 0) {
                union { uint2 u; uint16_t e[4]; } pk;
#pragma unroll
                for (int v = 0; v < 4; ++v) pk.e[v] = from_float<bf16_t>(activate(acc[i][j][v], act)).bits;
                *(uint2*)(orow + n) = pk.u;
            } else {
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (n + v < N) orow[n + v] = from_float<bf16_t>(activate(acc[i][j][v], act));
            }
        }
    }
}

// ------------------------------------------------------------------ products over the experts' rows (bfloat16, K a multiple of 64)
// Three kernels beside the one above, which keeps the heads' products of many rows and what these refuse.
//
// Few rows per expert (a decode step): what counts is the stream of the weights, and a stream needs work-groups enough to have tens of KB on their
// way from every compute unit.  A work-group owns a strip of 16 weight rows of one expert and up to 16 of its slots; its waves deal K out
// in steps of 64 (a lane fetches 32 bytes of its weight row and of its x row, a row's 128 bytes lie in one line; the order of k inside a step is
// the same for both operands and so does not matter), FEW_DEPTH steps on their way at once, and their sums meet in shared memory in the order of
// the waves.  Slots beyond the group's are copies of its last one and are not stored.
// HEADS: the same for groups that all have the step's rows (a head's columns of x and out a_group and out_group numbers apart), with a gate per output number:
// a decode step's products over heads, which one wave of the kernel above took whole (few work-groups, K one piece after the other).
#define FEW_DEPTH 4
struct HeadColumns {
    int a_group, out_group, rows;
    const bf16_t* gate;
    int gate_ld;
};

// This work-group's tile (blockIdx.y) among the groups' tiles of `height` rows, found by a prefix sum over the lanes: the group (-1: none), its tile's first row and the group's end.
struct GroupTile {
    int g, m0, m_end;
};
__device__ __forceinline__ GroupTile find_tile(const int* offsets, int groups, int height) {
    const int lane = threadIdx.x & 63;
    int first = 0;
    for (int base = 0; base < groups; base += TL_WAVE) {
        const int e = base + lane;
        const int from = e < groups ? offsets[e] : 0, to = e < groups ? offsets[e + 1] : 0;
        const int mine = (to - from + height - 1) / height;
        int upto = mine;
#pragma unroll
        for (int o = 1; o < TL_WAVE; o <<= 1) {
            const int t = __shfl_up(upto, o, TL_WAVE);
            if (lane >= o) upto += t;
        }
        const unsigned long long past = __ballot(first + upto > (int)blockIdx.y);
        if (past) {
            const int l = __builtin_amdgcn_readfirstlane(__ffsll(past) - 1);
            const int before = first + __builtin_amdgcn_readlane(upto, l) - __builtin_amdgcn_readlane(mine, l);
            return GroupTile{base + l, __builtin_amdgcn_readlane(from, l) + ((int)blockIdx.y - before) * height, __builtin_amdgcn_readlane(to, l)};
        }
        first += __builtin_amdgcn_readlane(upto, TL_WAVE - 1);
    }
    return GroupTile{-1, 0, 0};
}

template <int FEW_WAVES, bool HEADS>
__global__ void __launch_bounds__(FEW_WAVES * 64)
experts_few_rows_kernel(const bf16_t* __restrict__ a, int a_ld, const int* __restrict__ src, const bf16_t* __restrict__ w, bf16_t* __restrict__ out,
                        int out_ld, const int* __restrict__ offsets, int groups, int N, int K, int act, HeadColumns heads) {
    __shared__ __attribute__((aligned(16))) float red[FEW_WAVES][256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, kg = lane >> 4;
    const GroupTile tile = HEADS ? GroupTile{(int)blockIdx.z, (int)blockIdx.y * 16, heads.rows} : find_tile(offsets, groups, 16);
    const int g = tile.g, m0 = tile.m0, m_end = tile.m_end;
    if (g < 0) return;
    const int n0 = blockIdx.x * 16;
    const bf16_t* wrow = w + ((size_t)g * N + min(n0 + li, N - 1)) * K + 16 * kg;
    const int mine = min(m0 + li, m_end - 1);
    const bf16_t* xrow = a + (size_t)(!HEADS && src ? src[mine] : mine) * a_ld + (HEADS ? (size_t)g * heads.a_group : 0) + 16 * kg;
    f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int steps = K / 64;
    for (int s0 = wave; s0 < steps; s0 += FEW_WAVES * FEW_DEPTH) {
        Frag16 wf[FEW_DEPTH][2], xf[FEW_DEPTH][2];
#pragma unroll
        for (int u = 0; u < FEW_DEPTH; ++u) {
            const int k = min(s0 + u * FEW_WAVES, steps - 1) * 64;          // (beyond the end: fetched again, not used)
            wf[u][0].u = *(const uint4*)(wrow + k);
            wf[u][1].u = *(const uint4*)(wrow + k + 8);
            xf[u][0].u = *(const uint4*)(xrow + k);
            xf[u][1].u = *(const uint4*)(xrow + k + 8);
        }
#pragma unroll
        for (int u = 0; u < FEW_DEPTH; ++u) {
            if (s0 + u * FEW_WAVES < steps) {
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][0].v, xf[u][0].v, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[u][1].v, xf[u][1].v, acc, 0, 0, 0);
            }
        }
    }
    *(f32x4_t*)&red[wave][lane * 4] = acc;
    __syncthreads();
    if (wave > 0) return;
    f32x4_t sum = acc;
#pragma unroll
    for (int v = 1; v < FEW_WAVES; ++v) sum += *(const f32x4_t*)&red[v][lane * 4];
    // sum[v] = out[slot m0 + li][column n0 + 4 kg + v]
    const int m = m0 + li, n = n0 + 4 * kg, base_act = act & ~ACT_PAIRS;
    if (m >= m_end) return;
    bf16_t* orow = out + (size_t)m * out_ld + (HEADS ? (size_t)g * heads.out_group : 0);
    if (HEADS) {
        const bf16_t* grow = heads.gate ? heads.gate + (size_t)m * heads.gate_ld + (size_t)g * heads.out_group : nullptr;
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (n + v < N) orow[n + v] = from_float<bf16_t>(grow ? sum[v] * sigmoid(to_float(grow[n + v])) : sum[v]);
    } else if (act & ACT_PAIRS) {
#pragma unroll
        for (int v = 0; v < 4; v += 2)
            if (n + v + 1 < N) orow[(n + v) / 2] = from_float<bf16_t>(activate(sum[v], base_act) * sum[v + 1]);
    } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (n + v < N) orow[n + v] = from_float<bf16_t>(activate(sum[v], base_act));
    }
}

// Few rows per expert through rings in shared memory (see row_ring.h): a work-group owns rps weight rows of one expert (8 WJ at most) and 8 XH of its slots.
template <int WJ, int XH>
__global__ void __launch_bounds__(256)
experts_ring_kernel(const bf16_t* __restrict__ a, int a_ld, const int* __restrict__ src, const bf16_t* __restrict__ w, bf16_t* __restrict__ out, int out_ld,
                    const int* __restrict__ offsets, int groups, int N, int K, int act, int rps) {
    using S = RingShape<WJ, XH>;
    extern __shared__ __attribute__((aligned(16))) char ring[];
    const GroupTile tile = find_tile(offsets, groups, 8 * XH);
    if (tile.g < 0) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 15, kg = lane >> 4;
    const int n0 = blockIdx.x * rps, n_end = min(N, n0 + rps);
    unsigned woff[WJ], xoff[XH];
#pragma unroll
    for (int j = 0; j < XH; ++j) {
        const int r = 8 * (WJ + j) + lane / 8, c = (lane % 8) ^ ((r >> 1) & 7), slot = min(tile.m0 + r - 8 * WJ, tile.m_end - 1);
        xoff[j] = (unsigned)((src ? src[slot] : slot) * a_ld + c * 8) * 2;
    }
#pragma unroll
    for (int j = 0; j < WJ; ++j) {
        const int r = 8 * j + lane / 8, c = (lane % 8) ^ ((r >> 1) & 7);
        woff[j] = (unsigned)((min(n0 + r, n_end - 1) - n0) * K + c * 8) * 2;
    }
    ring_products<WJ, XH, 1>(w + ((size_t)tile.g * N + n0) * K, woff, a, xoff, K / 64, ring, wave, ring_spread(K));
    const int base_act = act & ~ACT_PAIRS;
    for (int q = wave; q < S::SH * S::MT; q += S::NW) {
        const int s = q / S::MT, t = q % S::MT, m = tile.m0 + 16 * t + li, n = n0 + 16 * s + 4 * kg;
        const f32x4_t sum = ring_sum<WJ, XH, 1>(ring, s, t);
        if (16 * t + li >= 8 * XH || m >= tile.m_end) continue;
        bf16_t* orow = out + (size_t)m * out_ld;
        if (act & ACT_PAIRS) {
#pragma unroll
            for (int v = 0; v < 4; v += 2)
                if (n + v + 1 < n_end) orow[(n + v) / 2] = from_float<bf16_t>(activate(sum[v], base_act) * sum[v + 1]);
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (n + v < n_end) orow[n + v] = from_float<bf16_t>(activate(sum[v], base_act));
        }
    }
}

// Many rows per expert (a prompt): the tile kernel with operands fetched straight into shared memory, over groups of rows.
static int experts_units = 256;       // compute units the tiles are dealt to
extern "C" void tl_experts_set_compute_units(int units) { if (units > 0) experts_units = units; }

struct ExpertsCall {
    const bf16_t* a;
    int a_ld;
    const int* src;
    const bf16_t* w;
    bf16_t* out;
    int out_ld;
    const int* offsets;
    int groups, rows, x_rows, N, K, act;      // rows: of out; x_rows: of a
};

static int launch_experts_few(const ExpertsCall& c, hipStream_t stream) {
    const dim3 grid((c.N + 15) / 16, c.rows / 16 + (c.groups < c.rows ? c.groups : c.rows));
    experts_few_rows_kernel<4, false><<<grid, 4 * 64, 0, stream>>>(c.a, c.a_ld, c.src, c.w, c.out, c.out_ld, c.offsets, c.groups, c.N, c.K, c.act, HeadColumns{});
    return TL_OK;
}

template <int WJ, int XH>
static int launch_experts_ring(const ExpertsCall& c, hipStream_t stream) {
    using S = RingShape<WJ, XH>;
    constexpr int rows = 8 * WJ;
    auto kernel = experts_ring_kernel<WJ, XH>;
    static hipError_t allowed = allow_lds(kernel, S::LDS);
    TL_REQUIRE(allowed == hipSuccess, "experts_ring: cannot get %zu bytes of shared memory", S::LDS);
    const dim3 grid((c.N + rows - 1) / rows, c.rows / (8 * XH) + (c.groups < c.rows ? c.groups : c.rows));
    kernel<<<grid, 256, S::LDS, stream>>>(c.a, c.a_ld, c.src, c.w, c.out, c.out_ld, c.offsets, c.groups, c.N, c.K, c.act, rows);
    return TL_OK;
}

template <int BM, int BN, int WGM, int WGN, int STAGES, bool PAIRS>
static int launch_experts_tile_t(const ExpertsCall& c, hipStream_t stream) {
    constexpr size_t lds = (size_t)STAGES * dl_slab_rows(BM, BN, WGM * WGN) * 64 * sizeof(bf16_t);
    auto kernel = gemm_dl_tile_kernel<BM, BN, WGM, WGN, STAGES, bf16_t, 0, ExpertRows<PAIRS>>;
    static hipError_t allowed = allow_lds(kernel, lds);
    if (allowed != hipSuccess) {
        tl_set_error("experts_tile: cannot get %zu bytes of shared memory: %s", lds, hipGetErrorString(allowed));
        return TL_ERR_HIP;
    }
    const long tiles = ((long)c.rows / BM + (c.groups < c.rows ? c.groups : c.rows)) * ((c.N + BN - 1) / BN);
    kernel<<<dim3(tiles), 64 * WGM * WGN, lds, stream>>>(c.a, c.w, nullptr, 0, c.out, 0, c.N, c.K, c.a_ld, c.out_ld, 0, 0,
                                                         ExpertRows<PAIRS>{c.offsets, c.src, c.groups, c.act});
    return TL_OK;
}

template <int BM, int BN, int WGM, int WGN, int STAGES>
static int launch_experts_tile(const ExpertsCall& c, hipStream_t stream) {
    return c.act & ACT_PAIRS ? launch_experts_tile_t<BM, BN, WGM, WGN, STAGES, true>(c, stream) : launch_experts_tile_t<BM, BN, WGM, WGN, STAGES, false>(c, stream);
}

enum ExpertsKernel { EX_RING_8, EX_FEW_4, EX_TILE_64x128, EX_TILE_128x128, EX_TILE_128x256, EX_TILE_256x256, EX_RING_16, EX_KERNELS };

static int launch_experts(int which, const ExpertsCall& c, hipStream_t stream) {
    int rc = TL_OK;
    switch (which) {
    case EX_RING_8: rc = launch_experts_ring<2, 1>(c, stream); break;
    case EX_RING_16: rc = launch_experts_ring<4, 2>(c, stream); break;
    case EX_FEW_4: rc = launch_experts_few(c, stream); break;
    case EX_TILE_64x128: rc = launch_experts_tile<64, 128, 1, 2, 3>(c, stream); break;
    case EX_TILE_128x128: rc = launch_experts_tile<128, 128, 2, 2, 2>(c, stream); break;
    case EX_TILE_128x256: rc = launch_experts_tile<128, 256, 2, 4, 3>(c, stream); break;
    case EX_TILE_256x256: rc = launch_experts_tile<256, 256, 2, 4, 2>(c, stream); break;
    default: TL_REQUIRE(false, "experts_gemm: no kernel %d", which);
    }
    if (rc != TL_OK) return rc;
    TL_CHECK_LAUNCH("experts_gemm");
    return TL_OK;
}

// Which kernel a call gets, by what the host knows: the slots of all groups together (how they are dealt to the groups only the GPU knows).
//
// Up to 12 slots a group on average (8 with K below 2048, where a wave has few slabs to keep on their way) the weights' stream sets the time: the rings, 16 weight rows and 8 slots a
// work-group up to 4 slots a group, 32 rows and 16 slots beyond; below 2048 columns of K and up to 4 slots a group the few-rows kernel, which has all its requests out at once.
// Measured (us; few rows with 8 waves / with 4 / rings of 16 rows and 8 slots / of 32 and 16 / tiles of 64 x 128; groups x N x K, every call on other weights):
//   16 x 2048 x 2048, 16 slots 19.8 / 21.8 / 18.5 / 18.6 / 28.4, 64 slots 28.1 / 30.8 / 24.4 / 25.4 / 37.2, 256 slots 44.0 / 44.0 / 38.5 / 29.2 / 37.0
//   16 x 2048 x 1024, 16 slots 18.1 / 11.1 / 12.1 / 11.4 / 14.1, 64 slots 26.5 / 15.3 / 16.1 / 15.3 / 16.0, 128 slots 28.6 / 17.4 / 18.1 / 15.7 / 16.2, 256 slots 41.9 / 23.5 / 27.0 / 18.9 / 16.6
//   32 x 4096 x 4096, 16 slots 76 / 81 / 75 / 81 / 83, 128 slots 181 / 187 / 170 / 175 / 180, 256 slots 209 / 211 / 194 / 176 / 181, 512 slots - / 308 / 262 / 197 / 182
//   32 x 4096 x 2048, 16 slots 43 / 43 / 39 / 41 / 55, 256 slots 113 / 115 / 104 / 90 / 119
//
// Beyond that, tiles: rounds of work-groups (two of the two smaller tiles to a compute unit) times a tile's time, fitted to single rounds at K of
// 1024 and 2048; every group ends in a tile that is half empty on average.  The figures were fitted to tiles of 32 x 32 x 16 products and hold for today's: over 37 sizes of 16 to 16384
// slots the kernel chosen takes 1.01 of the fastest one's time on average, 1.13 at most.  Measured (us; 64 x 128 / 128 x 128 / 128 x 256 / 256 x 256):
//   16 x 1024 x 2048, 2048 slots 33 / 35 / 34 / 46, 4096 slots 47 / 38 / 34 / 49, 16384 slots 119 / 103 / 90 / 101
//   16 x 2048 x 1024, 2048 slots 31 / 26 / 22 / 29, 4096 slots 45 / 44 / 39 / 32, 16384 slots 143 / 108 / 96 / 92
//   32 x 4096 x 4096, 2048 slots 228 / 190 / 190 / 250, 16384 slots 830 / 680 / 587 / 613
static int pick_experts(const ExpertsCall& c) {
    const bool eights = c.rows / 8 + (c.groups < c.rows ? c.groups : c.rows) <= 65535;      // a launch has that many tiles of 8 slots (experts_fit has counted those of 16)
    if ((long)c.rows <= (c.K < 2048 ? 8L : 12L) * c.groups) return (long)c.rows > 4L * c.groups ? EX_RING_16 : c.K < 2048 ? EX_FEW_4 : eights ? EX_RING_8 : EX_RING_16;
    static const struct { int kernel, bm, bn, per_unit; double fixed, per_k; } tiles[] = {
        {EX_TILE_64x128, 64, 128, 2, 9e-6, 6.5e-6}, {EX_TILE_128x128, 128, 128, 2, 7e-6, 13e-6},
        {EX_TILE_128x256, 128, 256, 1, 8e-6, 10.2e-6}, {EX_TILE_256x256, 256, 256, 1, 9e-6, 20e-6}};       // seconds of a tile: fixed, and per 1024 columns of K
    int best = EX_TILE_64x128;
    double best_t = 1e30;
    for (const auto& t : tiles) {
        const long groups = c.groups < c.rows ? c.groups : c.rows;
        const long count = ((long)c.rows + groups * (t.bm / 2) + t.bm - 1) / t.bm * ((c.N + t.bn - 1) / t.bn), slots = (long)t.per_unit * experts_units;
        const double est = (double)((count + slots - 1) / slots) * (t.fixed + t.per_k * c.K / 1024.0);
        if (est < best_t) { best_t = est; best = t.kernel; }
    }
    return best;
}

static bool experts_fit(const ExpertsCall& c) {
    // (a lane's offset from the first row of x, and of w from its tile's, is kept in 32 bits)
    return c.K % 64 == 0 && c.a_ld % 8 == 0 && ((uintptr_t)c.a % 16) == 0 && ((uintptr_t)c.w % 16) == 0 && (long)c.x_rows * c.a_ld * 2 < (1L << 31) &&
           256L * c.K * 2 < (1L << 31) && (long)(c.rows / 16 + c.groups) <= 65535;
}

// The kernel that a call of fitting operands gets, by its number (for tests).
extern "C" int tl_experts_choice(int groups, int rows, int N, int K) {
    ExpertsCall c{};
    c.groups = groups; c.rows = rows; c.N = N; c.K = K;
    return pick_experts(c);
}

// One kernel of ExpertsKernel by its number (tests cover each; tuning times them).
extern "C" int tl_experts_variant(const void* a, int a_ld, const void* src, const void* w, void* out, int out_ld, const void* offsets, int groups, int rows,
                                  int x_rows, int N, int K, int act, int which, hipStream_t stream) {
    const ExpertsCall c{(const bf16_t*)a, a_ld, (const int*)src, (const bf16_t*)w, (bf16_t*)out, out_ld, (const int*)offsets, groups, rows, x_rows, N, K, act};
    TL_REQUIRE(groups > 0 && rows > 0 && N > 0 && K > 0 && offsets && known_activation(act) && (!(act & ACT_PAIRS) || N % 2 == 0) && experts_fit(c), "experts_variant: bad arguments");
    return launch_experts(which, c, stream);
}

// Whether products over heads go to the few-rows kernel: up to eight of its work-groups to a compute unit, 64 rows at most (beyond, every strip of 16 rows reads the
// weights again).  Measured against the kernel without shared memory (us; heads x N x K): 32 x 512 x 128, 1 row 4.2 / 6.4, 32 rows 8.1 / 8.8, 48 rows (twelve to a
// unit) 10.9 / 8.9; 32 x 128 x 512, 1 row 3.8 / 11.1, 64 rows 9.7 / 15.4; 16 x 512 x 128, 64 rows 8.1 / 8.9; 8 x 192 x 64, 1 row 2.4 / 4.5.
static bool heads_few_rows(int rows, int groups, int N, int K) {
    return K % 64 == 0 && rows <= 64 && groups <= 65535 && (long)((N + 15) / 16) * ((rows + 15) / 16) * groups <= 8L * experts_units;
}

extern "C" int tl_grouped_gemm(const void* a, int a_ld, int a_group, const void* src, const void* w, void* out, int out_ld, int out_group,
                               const void* offsets, int groups, int rows, int x_rows, int N, int K, int act, const void* gate, int gate_ld, int dtype, int general,
                               hipStream_t stream) {
    TL_REQUIRE(groups > 0 && rows >= 0 && x_rows >= 0 && N > 0 && K > 0 && a_ld > 0 && out_ld > 0, "grouped_gemm: bad sizes");
    TL_REQUIRE(known_activation(act), "grouped_gemm: unknown activation %d", act);
    TL_REQUIRE(!(act & ACT_PAIRS) || (N % 2 == 0 && out_group == 0), "grouped_gemm: an activation in pairs needs an even number of columns");
    TL_REQUIRE(!gate || (!offsets && act == ACT_NONE && gate_ld >= (groups - 1) * out_group + N), "grouped_gemm: a gate stands beside groups of equal rows, with a number per output column");
    if (rows == 0) return TL_OK;
    // with offsets, `rows` is the number of sorted slots in all groups together: every group may end in a partial tile
    dim3 grid(offsets ? (rows + GG_T - 1) / GG_T + groups : (rows + GG_T - 1) / GG_T, (N + GG_T - 1) / GG_T, offsets ? 1 : groups), block(256);
    const bool aligned = K % 32 == 0 && a_ld % 8 == 0 && a_group % 8 == 0 && ((uintptr_t)a % 16) == 0 && ((uintptr_t)w % 16) == 0 &&
                         ((uintptr_t)out % 8) == 0;
    const ExpertsCall experts{(const bf16_t*)a, a_ld, (const int*)src, (const bf16_t*)w, (bf16_t*)out, out_ld, (const int*)offsets, groups, rows, x_rows, N, K, act};
    if (dtype == TL_DT_BF16 && offsets && !general && experts_fit(experts)) return launch_experts(pick_experts(experts), experts, stream);
    if (dtype == TL_DT_BF16 && aligned && !general && !offsets && act == ACT_NONE && heads_few_rows(rows, groups, N, K)) {
        const HeadColumns heads{a_group, out_group, rows, (const bf16_t*)gate, gate_ld};
        const dim3 fgrid((N + 15) / 16, (rows + 15) / 16, groups);
        auto kernel = K >= 512 ? experts_few_rows_kernel<4, true> : experts_few_rows_kernel<2, true>;      // (two steps of 64 to a wave, where there are so many)
        kernel<<<fgrid, K >= 512 ? 256 : 128, 0, stream>>>((const bf16_t*)a, a_ld, nullptr, (const bf16_t*)w, (bf16_t*)out, out_ld, nullptr, groups, N, K, act, heads);
        TL_CHECK_LAUNCH("heads_few_rows");
        return TL_OK;
    }
    if (dtype == TL_DT_BF16 && aligned && !general) {
        dim3 mgrid(offsets ? (rows + GM_BM - 1) / GM_BM + groups : (rows + GM_BM - 1) / GM_BM, (N + GM_BN - 1) / GM_BN, offsets ? 1 : groups);
        grouped_gemm_mfma_kernel<<<mgrid, block, 0, stream>>>((const bf16_t*)a, a_ld, a_group, (const int*)src, (const bf16_t*)w, (bf16_t*)out, out_ld,
                                                              out_group, (const int*)offsets, groups, rows, N, K, act, (const bf16_t*)gate, gate_ld);
        TL_CHECK_LAUNCH("grouped_gemm_mfma");
        return TL_OK;
    }
    if (dtype == TL_DT_F32)
        grouped_gemm_kernel<float><<<grid, block, 0, stream>>>((const float*)a, a_ld, a_group, (const int*)src, (const float*)w, (float*)out, out_ld,
                                                               out_group, (const int*)offsets, groups, rows, N, K, act, (const float*)gate, gate_ld);
    else if (dtype == TL_DT_BF16)
        grouped_gemm_kernel<bf16_t><<<grid, block, 0, stream>>>((const bf16_t*)a, a_ld, a_group, (const int*)src, (const bf16_t*)w, (bf16_t*)out, out_ld,
                                                                out_group, (const int*)offsets, groups, rows, N, K, act, (const bf16_t*)gate, gate_ld);
    else TL_REQUIRE(false, "grouped_gemm: unknown dtype %d", dtype);
    TL_CHECK_LAUNCH("grouped_gemm");
    return TL_OK;
}

// ------------------------------------------------------------------ the router's choice
// Per token (one wave): the `top` best of its `experts` outputs, best first (the lower index wins a tie), and their weights.
//   mode 0: the choice goes by the logits; the weights are the softmax over the chosen logits alone.
//   mode 1: the scores are the softmax over all logits; the choice goes by score + bias[e] (bias optional), the weights are the
//           chosen experts' scores as they are.
//   mode 2: the scores are the logits' sigmoids; the choice goes by score + bias[e] (bias optional), the weights are the chosen
//           experts' scores divided by their sum plus weight_eps.
// In every mode the weights are multiplied by weight_scale at the end.  group_size > 0: the experts lie in groups of that many neighbours, a
// group counts as much as the best of its experts (by what the choice goes by), and only the group_keep best groups' experts can be chosen.
struct RouteRule {
    int experts, top, mode;
    const float* bias;
    float weight_scale, weight_eps;
    int group_size, group_keep;
};

// One token's choice by one wave: z its logits, chosen and weights its `top` places.
__device__ __forceinline__ void route_token(const float* z, const RouteRule& r, int* chosen, float* weights) {
    const int lane = threadIdx.x % TL_WAVE, experts = r.experts, mode = r.mode;
    const float* bias = r.bias;
    float zmax = 0.f, den = 1.f;
    if (mode == 1) {
        float mx = -INFINITY;
        for (int e = lane; e < experts; e += TL_WAVE) mx = fmaxf(mx, z[e]);
        zmax = wave_max(mx);
        float sum = 0.f;
        for (int e = lane; e < experts; e += TL_WAVE) sum += expf(z[e] - zmax);
        den = wave_sum(sum);
    }
    float first = 0.f, sum = 0.f, mine = 0.f;           // lane j keeps the j-th choice's term
    // the best of this token's experts whose bit in `skip` (bit i: this lane's expert lane + 64 * i) is not set: its index, what it is chosen by, its score
    auto pick = [&](unsigned long long skip, float& best, float& score) {
        best = -INFINITY;
        score = 0.f;
        int at = 0x7fffffff;
        for (int e = lane, i = 0; e < experts; e += TL_WAVE, ++i) {
            float v = z[e], sc = 0.f;
            if (mode == 1) { sc = expf(v - zmax) / den; v = bias ? sc + bias[e] : sc; }
            else if (mode == 2) { sc = 1.f / (1.f + expf(-v)); v = bias ? sc + bias[e] : sc; }
            if (!((skip >> i) & 1ull) && (v > best || (v == best && e < at))) { best = v; at = e; score = sc; }
        }
#pragma unroll
        for (int o = TL_WAVE / 2; o > 0; o >>= 1) {
            const float ob = __shfl_xor(best, o, TL_WAVE);
            const float os = __shfl_xor(score, o, TL_WAVE);
            const int oa = __shfl_xor(at, o, TL_WAVE);
            if (ob > best || (ob == best && oa < at)) { best = ob; at = oa; score = os; }
        }
        return min(at, experts - 1);                    // (outputs that are no numbers choose nothing: the last expert stands in)
    };
    unsigned long long taken = 0;                       // the experts that are chosen already, or whose group is not kept
    if (r.group_size > 0) {
        unsigned long long kept = 0;                    // the best expert outside the kept groups tells the next best group
        for (int j = 0; j < r.group_keep; ++j) {
            float best, score;
            const int g = pick(kept, best, score) / r.group_size;
            for (int e = lane, i = 0; e < experts; e += TL_WAVE, ++i)
                if (e / r.group_size == g) kept |= 1ull << i;
        }
        taken = ~kept;
    }
    for (int j = 0; j < r.top; ++j) {
        float best, score;
        const int at = pick(taken, best, score);
        if (at % TL_WAVE == lane) taken |= 1ull << (at / TL_WAVE);
        if (j == 0) first = best;
        const float p = mode != 0 ? score : expf(best - first);
        sum += p;
        if (lane == j) { chosen[j] = at; mine = p; }
    }
    if (lane < r.top) weights[lane] = (mode == 1 ? mine : mode == 2 ? mine / (sum + r.weight_eps) : mine / sum) * r.weight_scale;
}

// The same for up to 64 experts, one to a lane: what the choice goes by stays in a register, and the best lane is found by its value's maximum and a ballot (the lowest lane of
// those that have it), where the walk above carries value, score and index through every exchange.  The same choices and weights, to the bit.
__device__ __forceinline__ void route_token_lanes(const float* z, const RouteRule& r, int* chosen, float* weights) {
    const int lane = threadIdx.x % TL_WAVE, experts = r.experts, mode = r.mode;
    const bool real = lane < experts;
    const float mine_z = real ? z[lane] : -INFINITY;
    float v = mine_z, score = 0.f;
    if (mode == 1) {
        const float zmax = wave_max(fmaxf(-INFINITY, mine_z));
        const float den = wave_sum(real ? expf(mine_z - zmax) : 0.f);
        score = expf(mine_z - zmax) / den;
    } else if (mode == 2) {
        score = 1.f / (1.f + expf(-mine_z));
    }
    if (mode != 0) v = r.bias && real ? score + r.bias[lane] : score;
    bool open = real && v == v;                         // (an output that is no number is not chosen)
    auto pick = [&](bool among, float& best, float& s) {
        best = wave_max(among ? v : -INFINITY);
        const unsigned long long have = __ballot(among && v == best);
        const int at = have ? __builtin_amdgcn_readfirstlane(__ffsll(have) - 1) : experts - 1;      // (none: the last expert stands in)
        s = have ? __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(score), at)) : 0.f;
        return at;
    };
    if (r.group_size > 0) {
        bool kept = false;
        for (int j = 0; j < r.group_keep; ++j) {
            float best, s;
            const int g = pick(open && !kept, best, s) / r.group_size;
            kept = kept || lane / r.group_size == g;
        }
        open = open && kept;
    }
    float first = 0.f, sum = 0.f, mine = 0.f;
    int mine_at = 0;
    for (int j = 0; j < r.top; ++j) {
        float best, s;
        const int at = pick(open, best, s);
        if (lane == at) open = false;
        if (j == 0) first = best;
        const float p = mode != 0 ? s : expf(best - first);
        sum += p;
        if (lane == j) { mine_at = at; mine = p; }
    }
    if (lane < r.top) {
        chosen[lane] = mine_at;
        weights[lane] = (mode == 1 ? mine : mode == 2 ? mine / (sum + r.weight_eps) : mine / sum) * r.weight_scale;
    }
}

__global__ void route_topk_kernel(const float* __restrict__ logits, RouteRule rule, int* __restrict__ chosen, float* __restrict__ weights, int tokens) {
    const int t = blockIdx.x * (blockDim.x / TL_WAVE) + threadIdx.x / TL_WAVE;
    if (t >= tokens) return;
    if (rule.experts <= TL_WAVE) route_token_lanes(logits + (size_t)t * rule.experts, rule, chosen + (size_t)t * rule.top, weights + (size_t)t * rule.top);
    else route_token(logits + (size_t)t * rule.experts, rule, chosen + (size_t)t * rule.top, weights + (size_t)t * rule.top);
}

// Sort of the (token, choice) pairs by expert, by one work-group: offsets[e] .. offsets[e + 1] - 1 are the slots of
// expert e, slot_token[slot] the token a slot reads, pair_slot[token * top + j] where the pair's output row lies.  cursor: [experts + 1] in shared memory.
__device__ __forceinline__ void route_sort(const int* chosen, int pairs, int top, int experts, int* cursor, int* __restrict__ offsets, int* __restrict__ slot_token,
                                           int* __restrict__ pair_slot) {
    for (int e = threadIdx.x; e <= experts; e += blockDim.x) cursor[e] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < pairs; i += blockDim.x) atomicAdd(&cursor[chosen[i] + 1], 1);
    __syncthreads();
    if (threadIdx.x < TL_WAVE) {                        // running sums, 64 experts at a time
        int before = 0;
        for (int base = 0; base < experts; base += TL_WAVE) {
            const int e = base + (int)threadIdx.x;
            int upto = e < experts ? cursor[e + 1] : 0;
#pragma unroll
            for (int o = 1; o < TL_WAVE; o <<= 1) {
                const int t = __shfl_up(upto, o, TL_WAVE);
                if ((int)threadIdx.x >= o) upto += t;
            }
            upto += before;
            if (e < experts) {
                cursor[e + 1] = upto;
                offsets[e + 1] = upto;
            }
            before = __shfl(upto, TL_WAVE - 1, TL_WAVE);
        }
        if (threadIdx.x == 0) offsets[0] = 0;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < pairs; i += blockDim.x) {
        const int slot = atomicAdd(&cursor[chosen[i]], 1);
        slot_token[slot] = i / top;
        pair_slot[i] = slot;
    }
}

__global__ void __launch_bounds__(1024)
route_sort_kernel(const int* __restrict__ chosen, int pairs, int top, int experts, int* __restrict__ offsets, int* __restrict__ slot_token, int* __restrict__ pair_slot) {
    extern __shared__ int cursor[];                     // [experts + 1]
    route_sort(chosen, pairs, top, experts, cursor, offsets, slot_token, pair_slot);
}

// Choice and sort of a decode step's tokens in one launch: a wave to a token, the choices stay in shared memory.  Both are chains of exchanges that hardly touch memory: what
// counts is their length and the launches (us: two kernels, each exchange with value, score and index, a running sum by one thread / this; 8 tokens, 2 of 16 by their logits 5.2 / 3.0,
// 2 of 18 by biased softmax 6.3 / 3.4, 4 of 32 by sigmoid 7.8 / 3.9, 2 of 16 in 4 groups 8.3 / 4.1).  Beyond 16 tokens the waves of one work-group would take turns: 32 tokens, 4 of 32
// 6.3 in one launch, 5.8 (at 64 tokens) in two.
#define ROUTE_FEW 16
__global__ void __launch_bounds__(1024)
route_few_kernel(const float* __restrict__ logits, RouteRule rule, float* __restrict__ weights, int tokens, int* __restrict__ offsets, int* __restrict__ slot_token,
                 int* __restrict__ pair_slot) {
    extern __shared__ int cursor[];                     // [experts + 1], then the choices [tokens * top]
    int* chosen = cursor + rule.experts + 1;
    const int t = threadIdx.x / TL_WAVE;                // (as many waves as tokens)
    route_token_lanes(logits + (size_t)t * rule.experts, rule, chosen + t * rule.top, weights + (size_t)t * rule.top);
    route_sort(chosen, tokens * rule.top, rule.top, rule.experts, cursor, offsets, slot_token, pair_slot);
}

extern "C" int tl_route(const void* logits, int tokens, int experts, int top, int mode, const void* bias, void* chosen, void* weights,
                        void* offsets, void* slot_token, void* pair_slot, float weight_scale, float weight_eps, int groups, int groups_kept,
                        hipStream_t stream) {
    TL_REQUIRE(mode >= 0 && mode <= 2, "route: unknown mode %d", mode);
    TL_REQUIRE(tokens >= 0 && experts > 0 && top > 0 && top <= experts && top <= TL_WAVE && experts <= 64 * TL_WAVE, "route: bad sizes (experts %d, top %d)", experts, top);
    TL_REQUIRE((experts + 1) * sizeof(int) <= 64 * 1024, "route: too many experts (%d)", experts);
    TL_REQUIRE(groups >= 0 && (groups == 0 || (experts % groups == 0 && groups_kept > 0 && groups_kept <= groups && top <= groups_kept * (experts / groups))),
               "route: %d of %d groups of %d experts do not hold %d choices", groups_kept, groups, experts, top);
    if (tokens == 0) return TL_OK;
    const RouteRule rule{experts, top, mode, (const float*)bias, weight_scale, weight_eps, groups > 0 ? experts / groups : 0, groups_kept};
    if (tokens <= ROUTE_FEW && experts <= TL_WAVE) {
        route_few_kernel<<<1, tokens * TL_WAVE, (experts + 1 + tokens * top) * sizeof(int), stream>>>((const float*)logits, rule, (float*)weights, tokens, (int*)offsets,
                                                                                                  (int*)slot_token, (int*)pair_slot);
        TL_CHECK_LAUNCH("route_few");
        return TL_OK;
    }
    route_topk_kernel<<<(tokens + 3) / 4, 4 * TL_WAVE, 0, stream>>>((const float*)logits, rule, (int*)chosen, (float*)weights, tokens);
    TL_CHECK_LAUNCH("route_topk");
    route_sort_kernel<<<1, 1024, (experts + 1) * sizeof(int), stream>>>((const int*)chosen, tokens * top, top, experts, (int*)offsets,
                                                                       (int*)slot_token, (int*)pair_slot);
    TL_CHECK_LAUNCH("route_sort");
    return TL_OK;
}

// ------------------------------------------------------------------ weighted sum of the chosen experts' outputs
// out[t, :] = sum_j weights[t, j] * y[pair_slot[t * top + j], :], summed in the order of the choices.  With `x`: a pair whose slot is
// offsets[real] or later chose an expert without tensors (an identity expert), and x[t, :] stands in for its row of y.  With `addend`
// (a shared expert's output): out[t, :] += addend[t, :], added last, in float.
template <typename T>
__global__ void combine_kernel(const T* __restrict__ y, const int* __restrict__ pair_slot, const float* __restrict__ weights,
                               T* __restrict__ out, const T* __restrict__ x, const int* __restrict__ offsets, int real, int top, int width,
                               const T* __restrict__ addend) {
    const int t = blockIdx.x;
    const int own_from = x ? offsets[real] : 0x7fffffff;
    for (int i = threadIdx.x; i < width; i += blockDim.x) {
        float a = 0.f;
        for (int j = 0; j < top; ++j) {
            const int slot = pair_slot[(size_t)t * top + j];
            const float v = slot >= own_from ? to_float(x[(size_t)t * width + i]) : to_float(y[(size_t)slot * width + i]);
            a = fmaf(weights[(size_t)t * top + j], v, a);
        }
        if (addend) a += to_float(addend[(size_t)t * width + i]);
        out[(size_t)t * width + i] = from_float<T>(a);
    }
}

// The same, 16 bytes of a row to a thread and four choices requested before the first is added (the sums keep their order): a number at a time every choice was a
// trip to memory of its own (eight tokens, 8 choices 7.9 -> 4.6 us on average; over a pass of prompts of 4 x 1100 tokens, 6 choices and a shared expert, and
// decoded tokens 33 -> 7.3).
template <typename T>
__global__ void __launch_bounds__(128)
combine_pieces_kernel(const T* __restrict__ y, const int* __restrict__ pair_slot, const float* __restrict__ weights, T* __restrict__ out, const T* __restrict__ x,
                      const int* __restrict__ offsets, int real, int top, int width, const T* __restrict__ addend) {
    constexpr int VEC = 16 / sizeof(T);
    struct __attribute__((aligned(16))) Piece { T v[VEC]; };
    const int t = blockIdx.x, i = (blockIdx.y * 128 + threadIdx.x) * VEC;
    if (i >= width) return;
    const int own_from = x ? offsets[real] : 0x7fffffff;
    const int* slots = pair_slot + (size_t)t * top;
    const float* w = weights + (size_t)t * top;
    auto row = [&](int slot) { return *(const Piece*)((slot >= own_from ? x + (size_t)t * width : y + (size_t)slot * width) + i); };
    Piece last;
    if (addend) last = *(const Piece*)(addend + (size_t)t * width + i);
    float a[VEC] = {};
    int j = 0;
    for (; j + 4 <= top; j += 4) {
        Piece p[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) p[u] = row(slots[j + u]);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int v = 0; v < VEC; ++v) a[v] = fmaf(w[j + u], to_float(p[u].v[v]), a[v]);
    }
    for (; j < top; ++j) {
        const Piece p = row(slots[j]);
#pragma unroll
        for (int v = 0; v < VEC; ++v) a[v] = fmaf(w[j], to_float(p.v[v]), a[v]);
    }
    Piece o;
#pragma unroll
    for (int v = 0; v < VEC; ++v) o.v[v] = from_float<T>(addend ? a[v] + to_float(last.v[v]) : a[v]);
    *(Piece*)(out + (size_t)t * width + i) = o;
}

// Rows of whole 16-byte pieces on 16 bytes; others keep the kernel of single numbers.
template <typename T>
static void launch_combine(const T* y, const int* pair_slot, const float* weights, T* out, const T* x, const int* offsets, int real, int tokens, int top, int width,
                           const T* addend, hipStream_t stream) {
    constexpr int VEC = 16 / sizeof(T);
    if (width % VEC == 0 && (((uintptr_t)y | (uintptr_t)out | (uintptr_t)x | (uintptr_t)addend) & 15) == 0 && width / VEC <= 128 * 65535)
        combine_pieces_kernel<T><<<dim3(tokens, (width / VEC + 127) / 128), 128, 0, stream>>>(y, pair_slot, weights, out, x, offsets, real, top, width, addend);
    else combine_kernel<T><<<tokens, 256, 0, stream>>>(y, pair_slot, weights, out, x, offsets, real, top, width, addend);
}

extern "C" int tl_combine(const void* y, const void* pair_slot, const void* weights, void* out, const void* x, const void* offsets, int real,
                          int tokens, int top, int width, const void* addend, int dtype, hipStream_t stream) {
    TL_REQUIRE(tokens >= 0 && top > 0 && width > 0 && real >= 0 && (!x || offsets), "combine: bad sizes");
    if (tokens == 0) return TL_OK;
    if (dtype == TL_DT_F32)
        launch_combine<float>((const float*)y, (const int*)pair_slot, (const float*)weights, (float*)out, (const float*)x, (const int*)offsets, real, tokens, top, width,
                              (const float*)addend, stream);
    else if (dtype == TL_DT_BF16)
        launch_combine<bf16_t>((const bf16_t*)y, (const int*)pair_slot, (const float*)weights, (bf16_t*)out, (const bf16_t*)x, (const int*)offsets, real, tokens, top,
                               width, (const bf16_t*)addend, stream);
    else TL_REQUIRE(false, "combine: unknown dtype %d", dtype);
    TL_CHECK_LAUNCH("combine");
    return TL_OK;
}

// ------------------------------------------------------------------ elementwise activation, in place
template <typename T>
__global__ void activation_kernel(T* __restrict__ x, size_t n, int act) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        x[i] = from_float<T>(activate(to_float(x[i]), act));
}

// The same in whole pieces of 16 bytes, one to a thread: bound by its bytes on prompts, where number by number it was bound by its requests (2048 x 8192 bfloat16
// numbers, 67 MB: 22.5 us before, 17.1 now).  ACT as a constant: one switch for the launch.
template <typename T, int ACT>
__global__ void __launch_bounds__(256) activation_pieces_kernel(T* __restrict__ x, size_t pieces) {
    constexpr int V = 16 / sizeof(T);
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= pieces) return;
    uint4 raw = *(const uint4*)(x + i * V);
    T* v = (T*)&raw;
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = from_float<T>(activate(to_float(v[e]), ACT));
    *(uint4*)(x + i * V) = raw;
}

template <typename T>
static void launch_activation(T* x, size_t n, int act, hipStream_t stream) {
    const size_t pieces = n * sizeof(T) / 16, blocks = (pieces + 255) / 256;
    if (n * sizeof(T) % 16 == 0 && ((uintptr_t)x % 16) == 0 && blocks < (1UL << 31)) {
#define TL_ACT(A) activation_pieces_kernel<T, A><<<(unsigned)blocks, 256, 0, stream>>>(x, pieces)
        if (act == ACT_RELU2) TL_ACT(ACT_RELU2);
        else if (act == ACT_SILU) TL_ACT(ACT_SILU);
        else if (act == ACT_GELU_TANH) TL_ACT(ACT_GELU_TANH);
        else TL_ACT(ACT_GELU);
#undef TL_ACT
        return;
    }
    activation_kernel<T><<<(int)((n + 1023) / 1024 < 8192 ? (n + 1023) / 1024 : 8192), 256, 0, stream>>>(x, n, act);
}

extern "C" int tl_activation(void* x, long n, int act, int dtype, hipStream_t stream) {
    TL_REQUIRE(n >= 0 && known_activation(act) && !(act & ACT_PAIRS), "activation: bad arguments");
    if (n == 0 || act == ACT_NONE) return TL_OK;
    TL_REQUIRE(dtype == TL_DT_F32 || dtype == TL_DT_BF16, "activation: unknown dtype %d", dtype);
    if (dtype == TL_DT_F32) launch_activation((float*)x, (size_t)n, act, stream);
    else launch_activation((bf16_t*)x, (size_t)n, act, stream);
    TL_CHECK_LAUNCH("activation");
    return TL_OK;
}

// ------------------------------------------------------------------ a gate against a token's own row
// out[t, n] = act(z[t, n]) * table[ids[t], n]: z float [tokens, dim] (a projection of the stream), `table` a slice of a token table (rows
// table_ld numbers apart).
template <typename T>
__global__ void token_gate_kernel(const float* __restrict__ z, const int* __restrict__ ids, const T* __restrict__ table, int table_ld, int vocab,
                                  T* __restrict__ out, int dim, int total, int act) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total) return;
    const int t = i / dim, n = i % dim, id = ids[t];
    if (id < 0 || id >= vocab) return;
    out[i] = from_float<T>(activate(z[i], act) * to_float(table[(size_t)id * table_ld + n]));
}

extern "C" int tl_token_gate(const void* z, const void* ids, const void* table, int table_ld, int vocab, void* out, int tokens, int dim, int act,
                             int dtype, hipStream_t stream) {
    TL_REQUIRE(tokens >= 0 && dim > 0 && table_ld >= dim && vocab > 0 && (long)tokens * dim < (1L << 31), "token_gate: bad sizes");
    TL_REQUIRE(known_activation(act) && !(act & ACT_PAIRS), "token_gate: unknown activation %d", act);
    if (tokens == 0) return TL_OK;
    const int total = tokens * dim, grid = (total + 255) / 256;
    if (dtype == TL_DT_F32)
        token_gate_kernel<float><<<grid, 256, 0, stream>>>((const float*)z, (const int*)ids, (const float*)table, table_ld, vocab, (float*)out, dim, total, act);
    else if (dtype == TL_DT_BF16)
        token_gate_kernel<bf16_t><<<grid, 256, 0, stream>>>((const float*)z, (const int*)ids, (const bf16_t*)table, table_ld, vocab, (bf16_t*)out, dim, total, act);
    else TL_REQUIRE(false, "token_gate: unknown dtype %d", dtype);
    TL_CHECK_LAUNCH("token_gate");
    return TL_OK;
}
