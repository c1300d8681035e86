// Matrix products out[M, N] = x[M, K] * w[N, K]^T (+ bias[N]).
//
// Both operands are row-major with K contiguous, which is how activations and
// nn.Linear-layout weights are stored.  This file holds the general kernel: a 64x64 or 128x128
// tile, 256 threads with a 4x4 or 8x8 micro-tile each, products and sums in true 32-bit
// (v_fma_f32; no matrix-core instruction of reduced precision).  It is the matrix
// product of the 32-bit path and the fallback of the bfloat16 path for shapes that
// the matrix-core kernels refuse.  The sum over K runs in one fixed order for every
// output element, whatever M is, so a row's result does not depend on the batch.
#include "activation.h"
#include "row_ring.h"

// The compute units of the GPU the library runs on: the caller tells it once (tl_gemm_set_compute_units, from
// the device's properties); 256, the MI355X on which every plan below was measured, until it does.
static int g_compute_units = 256;
extern "C" void tl_gemm_set_compute_units(int n) { if (n > 0) g_compute_units = n; }
extern "C" int tl_gemm_compute_units() { return g_compute_units; }
#define TL_COMPUTE_UNITS g_compute_units


#define GT_K 16

// BT x BT tile, 256 threads with a (BT / 16) x (BT / 16) micro-tile each: 64 x 64 for small products,
// 128 x 128 (64 products per thread and K step against four 16-byte reads of shared memory) for
// large ones.  Both add the products of an output element in the same order, k = 0, 1, 2, ...
template <typename TIn, typename TOut, int BT>
__global__ __launch_bounds__(256) void gemm_tile_kernel(const TIn* __restrict__ x, const TIn* __restrict__ w,
                                                        const void* __restrict__ bias, int bias_f32,
                                                        TOut* __restrict__ out, int M, int N, int K,
                                                        int ldx, int ldo) {
    constexpr int MT = BT / 16;                     // micro-tile edge
    constexpr int PER = BT * GT_K / 256;            // elements of each operand a thread loads per K step
    __shared__ float xs[GT_K][BT + 4];
    __shared__ float ws[GT_K][BT + 4];
    const int m0 = blockIdx.y * BT, n0 = blockIdx.x * BT;
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    // loaders: BT rows x 16 k per operand, PER consecutive k per thread
    const int lrow = threadIdx.x / (GT_K / PER);
    const int lk = (threadIdx.x % (GT_K / PER)) * PER;
    float acc[MT][MT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = 0.f;

    for (int k0 = 0; k0 < K; k0 += GT_K) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int k = k0 + lk + i;
            const int m = m0 + lrow, n = n0 + lrow;
            xs[lk + i][lrow] = (m < M && k < K) ? to_float(x[(size_t)m * ldx + k]) : 0.f;
            ws[lk + i][lrow] = (n < N && k < K) ? to_float(w[(size_t)n * K + k]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < GT_K; ++k) {
            float a[MT], b[MT];
#pragma unroll
            for (int i = 0; i < MT; ++i) a[i] = xs[k][ty * MT + i];
#pragma unroll
            for (int j = 0; j < MT; ++j) b[j] = ws[k][tx * MT + j];
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < MT; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int m = m0 + ty * MT + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const int n = n0 + tx * MT + j;
            if (n >= N) continue;
            float v = acc[i][j];
            if (bias) v += load_vec(bias, bias_f32, n);
            out[(size_t)m * ldo + n] = from_float<TOut>(v);
        }
    }
}

template <typename TIn, typename TOut>
static void launch_gemm_tile(const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int N, int K,
                             int ldx, int ldo, hipStream_t stream) {
    if (M >= 128 && N >= 128) {
        dim3 grid((N + 127) / 128, (M + 127) / 128), block(256);
        gemm_tile_kernel<TIn, TOut, 128><<<grid, block, 0, stream>>>((const TIn*)x, (const TIn*)w, bias, bias_f32, (TOut*)out, M, N, K, ldx, ldo);
    } else {
        dim3 grid((N + 63) / 64, (M + 63) / 64), block(256);
        gemm_tile_kernel<TIn, TOut, 64><<<grid, block, 0, stream>>>((const TIn*)x, (const TIn*)w, bias, bias_f32, (TOut*)out, M, N, K, ldx, ldo);
    }
}

// dtype: of x and w.  out_f32: write 32-bit results (logits) whatever the input dtype.
extern "C" int tl_gemm_general(const void* x, const void* w, const void* bias, int bias_f32, void* out,
                               int M, int N, int K, int ldx, int ldo, int dtype, int out_f32,
                               hipStream_t stream) {
    TL_REQUIRE(M >= 0 && N > 0 && K > 0 && ldx >= K && ldo >= N, "gemm: bad sizes M=%d N=%d K=%d ldx=%d ldo=%d", M, N, K, ldx, ldo);
    if (M == 0) return TL_OK;
    if (dtype == TL_DT_F32) launch_gemm_tile<float, float>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, stream);
    else if (dtype == TL_DT_BF16 && out_f32) launch_gemm_tile<bf16_t, float>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, stream);
    else if (dtype == TL_DT_BF16) launch_gemm_tile<bf16_t, bf16_t>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, stream);
    else TL_REQUIRE(false, "gemm: unknown dtype %d", dtype);
    TL_CHECK_LAUNCH("gemm_general");
    return TL_OK;
}


// =====================================================================================
// True 32-bit, few rows (M <= 16): the decode step's products of the 32-bit engine.
//
// The tile kernel above computes a 64-row tile whatever M is; with one to sixteen rows the
// product is a stream of the weight matrix and wants nothing but loads in flight.  A wave owns
// two weight rows; its lanes walk them in 16-byte pieces (lane, lane + 64, ...), multiply each
// piece with the matching piece of every x row (GV_KC columns of x at a time wait in shared
// memory) and keep one partial sum per (x row, weight row); at the end the 64 partial sums are
// added up in a fixed butterfly order.  A row's result therefore depends on neither M nor the
// other rows, as in the tile kernel, but its rounding differs from the tile kernel's (another
// order of the same sum).  Needs K % 4 == 0 and 16-byte aligned rows.
//
// END (see F32Pairs): a wave's two rows are what a gate or a rotation joins, and its sums go on to that, with the bits that the kernels behind a plain product would leave (us, one row, two
// launches / one, profiled: query, key and value of 5 heads of 32 from 96 columns 5.7 / 4.5; gate and up of 2 x 200 x 96 4.8 / 3.2; and a launch's gap less).
#define GV_ROWS 8
#define F32_PLAIN 0
#define F32_GATE 1
#define F32_ROTATE 2
// Rows of the matrix by pairs: pair p is the rows a = p / span * 2 span + p % span and a + span.  The gate's: span outputs, the gate's rows and then the up rows, out[m, p] = act(a) * b.  The
// rotation's: span is half a head, the two elements that a frequency turns (queries and keys; values are as they are); queries go to out, keys and values to their pages.
struct F32Pairs {
    int count, span, act;
    const int* positions;      // [M]
    const float* inv_freq;     // [head_dim / 2]
    const int* token_req;      // [M] request of each row (null: no cache write)
    const int* block_table;    // [requests, bt_stride]
    float* k_plane;            // [pages, kv_heads, page, head_dim]
    float* v_plane;            // [pages, kv_heads, head_dim, page]
    int bt_stride, page, q_heads, kv_heads;
    __host__ __device__ int row(int p) const { return p / span * 2 * span + p % span; }
};
__device__ __forceinline__ float f32_gate(int act, float g, float u) { return (act == 1 ? fmaxf(g, 0.f) : act == 2 ? gelu_tanh(g) : g / (1.f + expf(-g))) * u; }
// Pair p's cosine and sine at position pos, made while the weights are on their way.
__device__ __forceinline__ float2 f32_turn(const F32Pairs& pa, int p, int pos) {
    const float angle = (float)pos * pa.inv_freq[min(p, pa.count - 1) % pa.span];
    return make_float2(cosf(angle), sinf(angle));
}
// Pair p of row m, at position pos of page `page`.
__device__ __forceinline__ void f32_turn_store(const F32Pairs& pa, int p, float y1, float y2, float2 turn, int m, int pos, int page, float* out, int ldo) {
    const int half = pa.span, head = p / half, j = p - head * half, hd = 2 * half;
    if (head < pa.q_heads + pa.kv_heads) rope_turn(y1, y2, turn.x, turn.y);
    if (head < pa.q_heads) {
        float* o = out + (size_t)m * ldo + head * hd + j;
        o[0] = y1;
        o[half] = y2;
    } else if (page != 0) {       // page 0 is the sentinel (a padding row's): never written
        const int off = pos % pa.page;
        const size_t base = ((size_t)page * pa.kv_heads + (head - pa.q_heads) % pa.kv_heads) * pa.page * hd;
        const bool key = head < pa.q_heads + pa.kv_heads;
        float* o = key ? pa.k_plane + base + (size_t)off * hd + j : pa.v_plane + base + (size_t)j * pa.page + off;
        o[0] = y1;
        o[(size_t)half * (key ? 1 : pa.page)] = y2;
    }
}
template <int MR, int END>
__global__ __launch_bounds__(256) void gemv_f32_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                       const void* __restrict__ bias, int bias_f32,
                                                       float* __restrict__ out, int M, int N, int K, int ldx, int ldo, F32Pairs pa) {
    constexpr int KC = MR >= 8 ? 512 : 1024;       // 32 KB of x at most; at eight rows the shorter chunk keeps the kernel to 128 registers
    __shared__ float4 xs[MR][KC / 4];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int n0 = blockIdx.x * GV_ROWS + wave * 2, pair = n0 / 2;
    const int first = END ? pa.row(min(pair, pa.count - 1)) : min(n0, N - 1), second = END ? first + pa.span : min(n0 + 1, N - 1);
    const float* wa = w + (size_t)first * K;                 // rows past the end: read the last row, write nothing
    const float* wb = w + (size_t)second * K;
    int pos = 0, page = 0;                                   // (lane m: row m's)
    if (END == F32_ROTATE) {
        const int row = min(lane, M - 1);
        pos = pa.positions[row];
        if (pa.k_plane) page = pa.block_table[(size_t)pa.token_req[row] * pa.bt_stride + pos / pa.page];
    }
    float acc[MR][2];
#pragma unroll
    for (int m = 0; m < MR; ++m) acc[m][0] = acc[m][1] = 0.f;

    // A lane's pieces of its two rows are lane, lane + 64, ...: IPC of them per chunk of x.  The pieces of the next
    // chunk are requested while this chunk's are multiplied, so the stream of weights does not stop at the barriers
    // around the copy of x (with the requests made inside a chunk only, every chunk began with an empty pipe: the
    // 7B's decode step in 32-bit 9.5 -> see the measurements).  A piece beyond the row's end is fetched from the
    // row's last piece and cleared.
    constexpr int IPC = KC / 4 / 64;
    const int all = K / 4;
    float4 ra[IPC], rb[IPC];
    auto fetch = [&](int j, int c) {
        const int cc = min(c, all - 1);
        ra[j] = *(const float4*)(wa + 4 * cc);
        rb[j] = *(const float4*)(wb + 4 * cc);
    };
#pragma unroll
    for (int j = 0; j < IPC; ++j) fetch(j, lane + 64 * j);
    const float2 turn = END == F32_ROTATE ? f32_turn(pa, pair, pos) : make_float2(0.f, 0.f);
    for (int k0 = 0; k0 < K; k0 += KC) {
        const int pieces = min(KC, K - k0) / 4;
        __syncthreads();
        for (int i = threadIdx.x; i < MR * (KC / 4); i += 256) {
            const int m = i / (KC / 4), c = i % (KC / 4);
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (m < M && c < pieces) v = *(const float4*)(x + (size_t)m * ldx + k0 + 4 * c);
            xs[m][c] = v;
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < IPC; ++j) {
            const int c = lane + 64 * j;
            float4 a = ra[j], b = rb[j];
            if (k0 + KC < K) fetch(j, (k0 + KC) / 4 + c);
            if (c >= pieces) a = b = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                const float4 xv = xs[m][c];
                acc[m][0] = fmaf(a.w, xv.w, fmaf(a.z, xv.z, fmaf(a.y, xv.y, fmaf(a.x, xv.x, acc[m][0]))));
                acc[m][1] = fmaf(b.w, xv.w, fmaf(b.z, xv.z, fmaf(b.y, xv.y, fmaf(b.x, xv.x, acc[m][1]))));
            }
            // (one piece's reads of x at a time: moved up across the pieces they take the kernel from 112 to 192
            // registers at eight rows, and half the waves fit a compute unit)
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int r = 0; r < 2; ++r) acc[m][r] = wave_sum(acc[m][r]);
    if constexpr (END != F32_PLAIN) {
        float y1 = 0.f, y2 = 0.f;                            // lane m has row m
#pragma unroll
        for (int m = 0; m < MR; ++m)
            if (lane == m) { y1 = acc[m][0]; y2 = acc[m][1]; }
        if (lane >= M || pair >= pa.count) return;
        if (bias) { y1 += load_vec(bias, bias_f32, first); y2 += load_vec(bias, bias_f32, second); }
        if constexpr (END == F32_GATE) out[(size_t)lane * ldo + pair] = f32_gate(pa.act, y1, y2);
        else f32_turn_store(pa, pair, y1, y2, turn, lane, pos, page, out, ldo);
        return;
    }
    if (lane < 2 && n0 + lane < N) {
        const int n = n0 + lane;
        const float b = bias ? load_vec(bias, bias_f32, n) : 0.f;
#pragma unroll
        for (int m = 0; m < MR; ++m)
            if (m < M) out[(size_t)m * ldo + n] = (lane ? acc[m][1] : acc[m][0]) + b;
    }
}

// The same on the matrix cores, 2 to 16 rows: v_mfma_f32_16x16x4_f32 multiplies and adds in true 32-bit (as
// v_mfma_f32_32x32x2_f32 below), and a step of several rows costs the stream of weights and little else, where the
// kernel above spends a multiply-add per row and weight (the dispatch takes this kernel from 9 rows on where K is no multiple of 32, which the rings want).  A work-group of eight waves owns 16 weight rows; chunks of GM_KC columns of x wait in shared
// memory (rows beyond M as zeros); within a chunk the waves take its pieces of 16 columns in turn.  A lane fetches
// four neighbouring k of its weight row and of its x row at once: lane group g = lane / 16 takes k = 4 g .. 4 g + 3
// of the piece, so instruction e of a piece multiplies k = 4 g + e of the four groups: which k meet in one instruction
// is free as long as both operands agree.  The pieces of the next chunk are requested while this chunk's are
// multiplied.  Each wave's sum over its pieces runs in one fixed order and the eight partial tiles are added in wave
// order, whatever M is: a row's result does not depend on the batch (it differs from the other 32-bit kernels' by
// rounding).  Needs K % 4 == 0 and 16-byte aligned rows.
typedef float gm_f32x4_t __attribute__((ext_vector_type(4)));
#define GM_WAVES 8
#define GM_KC 512                        // columns of x in shared memory at a time: 16 rows x 512 x 4 bytes = 32 KB
#define GM_LD (GM_KC + 4)                // floats between rows of x: 16-byte reads of 16 rows fall on all banks
__global__ __launch_bounds__(GM_WAVES * 64) void gemv_f32_mfma_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                      const void* __restrict__ bias, int bias_f32,
                                                                      float* __restrict__ out, int M, int N, int K, int ldx, int ldo) {
    __shared__ __attribute__((aligned(16))) float xs[16 * GM_LD];
    __shared__ __attribute__((aligned(16))) float red[GM_WAVES * 256];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int li = lane & 15, lg = lane >> 4;
    const int n0 = blockIdx.x * 16;
    const float* wrow = w + (size_t)min(n0 + li, N - 1) * K;       // rows past the end: the last row again, never stored
    constexpr int PPW = GM_KC / 16 / GM_WAVES;                     // pieces of 16 columns a wave takes of a chunk
    gm_f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
    float4 ring[PPW];
    // piece q of the chunk at k0 that is this wave's: columns k0 + 16 (wave + q GM_WAVES) + 4 lg .. + 3; beyond K the
    // row's last whole four are fetched and cleared
    auto fetch = [&](int q, int k0) {
        const int k = k0 + 16 * (wave + q * GM_WAVES) + 4 * lg;
        ring[q] = *(const float4*)(wrow + min(k, K - 4));
        if (k >= K) ring[q] = make_float4(0.f, 0.f, 0.f, 0.f);
    };
#pragma unroll
    for (int q = 0; q < PPW; ++q) fetch(q, 0);
    for (int k0 = 0; k0 < K; k0 += GM_KC) {
        const int cols = min(GM_KC, K - k0);
        __syncthreads();                                           // the chunk before is read
        for (int i = tid; i < 16 * (GM_KC / 4); i += GM_WAVES * 64) {
            const int m = i / (GM_KC / 4), c = i % (GM_KC / 4);
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (m < M && 4 * c < cols) v = *(const float4*)(x + (size_t)m * ldx + k0 + 4 * c);
            *(float4*)(&xs[m * GM_LD + 4 * c]) = v;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < PPW; ++q) {
            const float4 a = ring[q];
            if (k0 + GM_KC < K) fetch(q, k0 + GM_KC);
            const float4 b = *(const float4*)(&xs[li * GM_LD + 16 * (wave + q * GM_WAVES) + 4 * lg]);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, acc, 0, 0, 0);
        }
    }
    // a lane holds weight rows i = 4 (lane / 16) + v and x row j = lane % 16 of its wave's partial tile
    *(gm_f32x4_t*)(&red[(wave * 64 + lane) * 4]) = acc;
    __syncthreads();
    if (wave == 0) {
        gm_f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int wv = 0; wv < GM_WAVES; ++wv) sum += *(const gm_f32x4_t*)(&red[(wv * 64 + lane) * 4]);
        const int m = li;
        if (m < M) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int n = n0 + 4 * lg + v;
                if (n < N) out[(size_t)m * ldo + n] = sum[v] + (bias ? load_vec(bias, bias_f32, n) : 0.f);
            }
        }
    }
}

static bool gemv_f32_fits(const void* x, const void* w, int M, int K, int ldx) {
    return M <= 16 && K % 4 == 0 && ldx % 4 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0;
}

template <int END>
static void launch_gemv_f32_fma(const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int N, int K, int ldx, int ldo, const F32Pairs& pa, hipStream_t stream) {      // up to 8 rows
    dim3 grid((N + GV_ROWS - 1) / GV_ROWS), block(256);
#define GV_LAUNCH(MR) gemv_f32_kernel<MR, END><<<grid, block, 0, stream>>>((const float*)x, (const float*)w, bias, bias_f32, (float*)out, M, N, K, ldx, ldo, pa)
    if (M <= 1) GV_LAUNCH(1);
    else if (M <= 2) GV_LAUNCH(2);
    else if (M <= 4) GV_LAUNCH(4);
    else GV_LAUNCH(8);
#undef GV_LAUNCH
}

static void launch_gemv_f32_mfma(const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int N, int K, int ldx, int ldo, hipStream_t stream) {
    gemv_f32_mfma_kernel<<<dim3((N + 15) / 16), dim3(GM_WAVES * 64), 0, stream>>>((const float*)x, (const float*)w, bias, bias_f32, (float*)out, M, N, K, ldx, ldo);
}

// =====================================================================================
// True 32-bit on the matrix cores, more than 16 rows: the prompt steps of the 32-bit engine.
//
// v_mfma_f32_32x32x2_f32 and v_mfma_f32_16x16x4_f32 multiply 32-bit operands and add in 32-bit: they are no reduced-precision mode
// (nothing is rounded to a shorter format on the way), and they run at four times the rate of the
// v_fma_f32 tile kernel above.  A work-group of four waves owns a tile of 2 B FMB x 2 B FNB outputs, a wave
// FMB x FNB blocks of B x B of them.
//
// What bounds it is the matrix instruction (64 cycles for a block of 32, 32 for one of 16, against 8 of shared memory for a wave's 16-byte read), so all else has to
// stay out of its way: slabs of 32 columns of both operands go straight into shared memory, laid out and requested as in direct_tile.h (a row of a slab is 128 bytes
// there too), STAGES of them in flight or in use, and the operands of the next phase (PHASE times eight columns) are read while this one's are multiplied.  The last
// phase of a slab waits for the next slab and meets the other waves halfway through its products; behind that barrier go the first reads of the next slab and the
// requests into the buffer just given up.  Measured against slabs of 16 columns through registers with a barrier each (us; the matrix instruction's 157 TFLOP/s alone
// would take the last figure): 753 x 37888 x 3584 1772 -> 1443 (1303), 753 x 3584 x 18944 1098 -> 863 (651), 753 x 3584 x 3584 212 -> 166 (123), 301 x 37888 x 3584
// 832 -> 631 (521), 2048 x 2048 x 2048 167 -> 124 (109).  What is left is the last round of tiles and the clock.
//
// A lane holds four neighbouring k of its row: with blocks of 32 lanes 0-31 k = 8c .. 8c+3 and lanes 32-63 k = 8c+4 .. 8c+7 of a chunk of eight, so instruction e
// of a chunk multiplies k = 8c + e and 8c + 4 + e: which k meet in one instruction is free as long as both operands agree.  With blocks of 16 an instruction takes the k of two of these
// in the same order (8c, 8c + 4, 8c + 1, 8c + 5 and then the two further on), and its sums come out the same to the last bit.  The sum of an output element
// runs in that one fixed order whatever M is, whichever tile is taken and wherever the element lies in it, so a row's result does not depend on the batch; it differs from the
// other 32-bit kernels' by rounding (another order of the same sum).  Needs K % 4 == 0 and 16-byte aligned rows; what K has beyond whole slabs goes through
// registers, columns past K as zeros.
#define GF_TK 32
template <int B, int FMB, int FNB, int STAGES, int WAVES_PER_SIMD, int PHASE>
__global__ __launch_bounds__(256, WAVES_PER_SIMD) void gemm_f32_mfma_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                            const void* __restrict__ bias, int bias_f32,
                                                            float* __restrict__ out, int M, int N, int K, int ldx, int ldo) {
    constexpr int BM = 2 * B * FMB, BN = 2 * B * FNB, ROWS = BM + BN;
    constexpr int E = B == 32 ? 4 : 2, V = B * B / 64;      // instructions of a chunk and block, results of a lane and block
    typedef float sums_t __attribute__((ext_vector_type(V)));
    typedef float operand_t __attribute__((ext_vector_type(E)));
    constexpr int LOADS = ROWS / 32;                        // requests of a wave per slab: eight rows each, BM / 32 of them of x
    constexpr int SLAB = ROWS * GF_TK;                      // floats
    extern __shared__ __attribute__((aligned(16))) float gf_lds[];     // [STAGES][ROWS][GF_TK]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int lr = lane % B, lh = lane / B;

    // tile order as in direct_tile.h: each XCD walks 8 x 8 blocks of tiles out of its own L2
    int m0, n0;
    {
        const int tiles_n = gridDim.x, tiles_m = gridDim.y, total = tiles_n * tiles_m, id = blockIdx.y * tiles_n + blockIdx.x;
        const int xcd = id % 8, lid = xcd * (total / 8) + min(xcd, total % 8) + id / 8;
        const int per_group = 8 * tiles_n, first_m = (lid / per_group) * 8, rows = min(tiles_m - first_m, 8);
        m0 = (first_m + (lid % per_group) % rows) * BM;
        n0 = ((lid % per_group) / rows) * BN;
    }

    sums_t acc[FNB][FMB];
#pragma unroll
    for (int i = 0; i < FNB; ++i)
#pragma unroll
        for (int j = 0; j < FMB; ++j)
#pragma unroll
            for (int v = 0; v < V; ++v) acc[i][j][v] = 0.f;

    // request j of this wave fills the rows 8 (wave + 4 j) .. + 7 of the stacked [x rows; w rows] slab; piece c of row r lies in slot c ^ ((r >> 1) & 7).
    // Rows past the end read the last row (never stored).
    unsigned soff[LOADS];
    int ldst[LOADS];
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
        const int row = 8 * (wave + 4 * j) + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        soff[j] = j < BM / 32 ? (unsigned)((min(m0 + row, M - 1) - m0) * ldx + c * 4) * 4u : (unsigned)((min(n0 + row - BM, N - 1) - n0) * K + c * 4) * 4u;
        ldst[j] = __builtin_amdgcn_readfirstlane(8 * (wave + 4 * j) * GF_TK * 4);
    }
    const float *xt = x + (size_t)m0 * ldx, *wt = w + (size_t)n0 * K;
    const unsigned lds_base = (unsigned)(uintptr_t)((void __attribute__((address_space(3)))*)gf_lds);
    const int slabs = K / GF_TK, rest = K % GF_TK;

    // a chunk's operands (blocks are 16 or 32 rows apart, which leaves the slots' order as it is)
    const int x_at = (wm * B * FMB + lr) * GF_TK, w_at = (BM + wn * B * FNB + lr) * GF_TK, turn = (lr >> 1) & 7;
    operand_t a[2][PHASE][FNB], b[2][PHASE][FMB];
    auto read = [&](const float* slab, int phase, int set, int op) {
        const int h = op / (FMB + FNB), o = op % (FMB + FNB), c = phase * PHASE + h;
        const float* row = slab + (o < FNB ? w_at + o * B * GF_TK : x_at + (o - FNB) * B * GF_TK);
        operand_t& to = o < FNB ? a[set][h][o] : b[set][h][o - FNB];
        if constexpr (B == 32) {
            to = *(const operand_t*)(row + ((2 * c + lh) ^ turn) * 4);
        } else {
            const float* at = row + ((2 * c + (lh & 1)) ^ turn) * 4 + (lh >> 1);
            to[0] = at[0];
            to[1] = at[2];
        }
    };
    auto product = [&](int set, int q) {
        const int h = q / (E * FMB * FNB), e = q / (FMB * FNB) % E, i = q % (FMB * FNB) / FMB, j = q % FMB;
        if constexpr (B == 32) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[set][h][i][e], b[set][h][j][e], acc[i][j], 0, 0, 0);
        else acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[set][h][i][e], b[set][h][j][e], acc[i][j], 0, 0, 0);
    };
    static_assert(GF_TK / 8 / PHASE % 2 == 0, "two sets of operands in turn");
    constexpr int READS = PHASE * (FMB + FNB), PHASES = GF_TK / 8 / PHASE, NM = PHASE * E * FMB * FNB, BARRIER_AT = NM / 2;
    if (slabs > 0) {
        // (past the end the last slab is requested again, which nobody reads: the count of requests in flight is the same in every step)
        auto request = [&](int slab, int j) {
            load_to_lds_at((j < BM / 32 ? xt : wt) + min(slab, slabs - 1) * GF_TK, soff[j], lds_base + (slab % STAGES) * (SLAB * 4) + ldst[j]);
        };
#pragma unroll
        for (int st = 0; st < STAGES; ++st)
#pragma unroll
            for (int j = 0; j < LOADS; ++j) request(st, j);
        wait_direct_loads<(STAGES - 1) * LOADS>();
        __syncthreads();
#pragma unroll
        for (int op = 0; op < READS; ++op) read(gf_lds, 0, 0, op);
        __builtin_amdgcn_sched_barrier(0);
        for (int sl = 0; sl < slabs; ++sl) {
            const float *here = gf_lds + (sl % STAGES) * SLAB, *next = gf_lds + ((sl + 1) % STAGES) * SLAB;
#pragma unroll
            for (int c = 0; c < PHASES; ++c) {
                const bool last = c + 1 == PHASES;
                const int start = last ? BARRIER_AT : 0, ops = READS + (last ? LOADS : 0), per = (ops + NM - start - 1) / (NM - start);
                int op = 0;
#pragma unroll
                for (int q = 0; q < NM; ++q) {
                    if (last && q == start) {
                        wait_direct_loads<(STAGES - 2) * LOADS>();
                        __syncthreads();
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    product(c & 1, q);
                    __builtin_amdgcn_sched_barrier(0);
                    if (q < start) continue;
#pragma unroll
                    for (int e = 0; e < per; ++e, ++op) {
                        if (op < READS) read(last ? next : here, last ? 0 : c + 1, (c + 1) & 1, op);
                        else if (op < ops) request(sl + STAGES, op - READS);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        wait_direct_loads<0>();
    }
    if (rest) {
        __syncthreads();                                    // (all direct loads have landed and all operands are read)
#pragma unroll
        for (int j = 0; j < LOADS; ++j) {
            const int row = 8 * (wave + 4 * j) + (lane >> 3), piece = lane & 7, k = slabs * GF_TK + 4 * piece;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (k < K) v = *(const float4*)(row < BM ? x + (size_t)min(m0 + row, M - 1) * ldx + k : w + (size_t)min(n0 + row - BM, N - 1) * K + k);
            *(float4*)(gf_lds + row * GF_TK + ((piece ^ ((row >> 1) & 7)) * 4)) = v;
        }
        __syncthreads();
        for (int c = 0; 8 * PHASE * c < rest; ++c) {
#pragma unroll
            for (int op = 0; op < READS; ++op) read(gf_lds, c, 0, op);
#pragma unroll
            for (int q = 0; q < NM; ++q) product(0, q);
        }
    }
    // weight block times x block: a lane holds row m = lane % B of x and the output columns
    // n = 8 (v / 4) + 4 (lane / 32) + v % 4 of a 32 x 32 block, 4 (lane / 16) + v of a 16 x 16 block, four neighbours at a time
    const bool quads = N % 4 == 0 && ldo % 4 == 0 && ((uintptr_t)out % 16) == 0;
#pragma unroll
    for (int j = 0; j < FMB; ++j) {
        const int m = m0 + wm * B * FMB + j * B + lr;
        if (m >= M) continue;
#pragma unroll
        for (int i = 0; i < FNB; ++i)
#pragma unroll
            for (int g = 0; g < V / 4; ++g) {
                const int n = n0 + wn * B * FNB + i * B + 8 * g + 4 * lh;
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * g + e] + ((bias && n + e < N) ? load_vec(bias, bias_f32, n + e) : 0.f);
                if (quads) {
                    if (n < N) *(float4*)(out + (size_t)m * ldo + n) = make_float4(v[0], v[1], v[2], v[3]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (n + e < N) out[(size_t)m * ldo + n + e] = v[e];
                }
            }
    }
}

// (a lane's offset from its tile's first row is kept in 32 bits)
static bool gemm_f32_mfma_fits(const void* x, const void* w, int M, int K, int ldx) {
    return M > 16 && K >= 4 && K % 4 == 0 && ldx % 4 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0 && ldx < (1 << 22) && K < (1 << 22);
}

// The size of tiles of a 32-bit product: 1 64 x 64, 2 64 x 128, 3 128 x 128 of blocks of 32; 4 64 x 32 and 5 32 x 32 of blocks of 16, which move twice the operands per product
// but leave few rows against a narrow matrix more work-groups and a shorter chain each.
//
// Microseconds per column of K: a start and a round of work-groups, up to TL_COMPUTE_UNITS of them at once (the smaller tiles' rounds overlap on a unit).  Fitted to 17 to 2048
// rows against thirteen matrices 288 to 37888 wide, within a tenth of each; the sums are the same whichever is taken.  Measured (us; 64 x 64 / 64 x 128 / 128 x 128 / 64 x 32 / 32 x 32):
// 17 x 4608 x 3584 65 / 113 / 211 / 45 / 33, 100 x 3584 x 3584 66 / 114 / 214 / 45 / 52, 301 x 3584 x 18944 578 / 586 / 1111 / 600 / 659, 753 x 3584 x 18944 863 / 1084 / 1117 / 1191 / 1443,
// 753 x 4608 x 3584 225 / 210 / 216 / 267 / 350, 301 x 37888 x 3584 675 / 631 / 816 / 894 / 1164, 753 x 37888 x 3584 1618 / 1472 / 1443 / 2096 / 2744.
// A size whose rows of tiles are more than a launch has in y is not considered: beyond 4.19 million rows the tiles are 128 high.
extern "C" int tl_gemm_f32_tile(int M, int N) {
    static const struct { int bm, bn; double start, round; } sizes[] = {{64, 64, 0.002, 0.0155}, {64, 128, 0.001, 0.0293}, {128, 128, 0.003, 0.0573}, {64, 32, 0.002, 0.0105}, {32, 32, 0.0025, 0.0068}};
    double best = 1e30;
    int tile = 3;
    for (int t = 0; t < 5; ++t) {
        const long rows = ((long)M + sizes[t].bm - 1) / sizes[t].bm, tiles = rows * (((long)N + sizes[t].bn - 1) / sizes[t].bn);
        if (rows > 65535) continue;
        const double est = sizes[t].start + sizes[t].round * ((tiles + TL_COMPUTE_UNITS - 1) / TL_COMPUTE_UNITS);
        if (est < best) { best = est; tile = t + 1; }
    }
    return tile;
}

template <int B, int FMB, int FNB, int STAGES, int WAVES_PER_SIMD, int PHASE>
static void launch_gemm_f32_tile(const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int N, int K, int ldx, int ldo, hipStream_t stream) {
    constexpr int BM = 2 * B * FMB, BN = 2 * B * FNB;
    constexpr size_t lds = (size_t)STAGES * (BM + BN) * GF_TK * sizeof(float);
    static_assert(lds <= 65536, "no more shared memory than a kernel has unasked");
    gemm_f32_mfma_kernel<B, FMB, FNB, STAGES, WAVES_PER_SIMD, PHASE><<<dim3((N + BN - 1) / BN, (M + BM - 1) / BM), dim3(256), lds, stream>>>(
        (const float*)x, (const float*)w, bias, bias_f32, (float*)out, M, N, K, ldx, ldo);
}

// `tile`: 0 by the rule above, else one of its sizes (tests cover each; tuning times them).  Two work-groups of the larger tiles (64 and 48 KB) and three of 64 x 64 fit a compute unit.
static void launch_gemm_f32_mfma(const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int N, int K,
                                 int ldx, int ldo, hipStream_t stream, int tile = 0) {
    if (tile == 0) tile = tl_gemm_f32_tile(M, N);
    auto launch = tile == 1 ? launch_gemm_f32_tile<32, 1, 1, 3, 3, 2> : tile == 2 ? launch_gemm_f32_tile<32, 1, 2, 2, 2, 1> : tile == 3 ? launch_gemm_f32_tile<32, 2, 2, 2, 2, 1>
                : tile == 4 ? launch_gemm_f32_tile<16, 2, 1, 4, 3, 2> : launch_gemm_f32_tile<16, 1, 1, 6, 3, 2>;
    launch(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, stream);
}

// =====================================================================================
// bfloat16 on the matrix cores, few rows (M <= 64): the decode step's products.
//
// Such a product is a stream of the weight matrix through the chip once; the kernel is
// built so that nothing but HBM limits it.  out^T tile = W tile * x^T on
// v_mfma_f32_16x16x32_bf16: the A operand is 16 rows of W, the B operand 16 rows of x, both
// read straight from memory as 16-byte pieces of a K-contiguous row (no shared-memory
// staging, no barrier in the loop).  A wave owns R strips of 16 weight rows and MT tiles of
// 16 activation rows and walks K in steps of 64: lane group g = lane / 16 reads the 32
// contiguous bytes k = 64 s + 16 g .. + 16 of its row, so the four groups of a row consume
// one full 128-byte line; the two 16-byte halves feed two MFMAs (how k is dealt to lanes is
// free as long as A and B agree).  The KS waves of a work-group take the steps s = wave,
// wave + KS, ... and add their partial tiles through shared memory in a fixed order, so
// the result is deterministic.  One row of x is as good as free (the lanes of a wave that read the
// same address share the fetch); with more rows x costs M / 16 of the weight traffic again, so it is
// copied into shared memory (XL) by no more work-groups than the compute units hold at once, each
// of which then walks a run of outputs of its own, strip after strip, and requests the first
// steps of its next strip before it adds up the sums of this one (measured at M = 8, 7B sizes:
// gate/up 57 -> 51 us, LM head 207 -> 189 us).
// Needs K % 8 == 0 and 16-byte aligned rows; other shapes go to the general kernel.  Products with K a multiple of 64, which the figures here were measured on, are gemm_ring_kernel's by now but for:
// one row against more than 32768 columns, the products of one row that make their norm themselves, the slabs of one row against up to 4096 columns, projections with their rotation of 16384
// columns and more, gates of 2 to 16 rows with more than 16384 outputs and K below 1024.  The rules below (balanced_rows, plan_strips, pick_skinny, the copy of x) serve those and every other K.
#define SK_KOFF(lg) (16 * (lg))     // a lane reads 32 contiguous bytes per step (other splits measured the same)
#define SK_SECOND 8
#define SK_LOAD(p) (*(const uint4*)(p))

__device__ __forceinline__ void lds_barrier() {
    // waits for this wave's shared-memory traffic only: weight fetches stay in flight across it
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Register sets of weights a wave of the skinny kernel keeps in flight: as many K steps as fit
// beside the accumulators (a step takes 8 registers per strip and 8 per tile of activation rows).
template <int R, int MT, int KS>
constexpr int skinny_depth() {
    const int per_step = 8 * R + 8 * MT;
    const int budget = KS >= 16 ? 64 : 128;       // 1024 threads leave 128 registers a lane
    const int d = budget / per_step;
    return d < 2 ? 2 : (d > 8 ? 8 : d);
}

// SW (gate/up product with the SwiGLU gate applied to the accumulators): w holds blocks of 64
// rows, 32 gate rows followed by the 32 up rows of the same columns; a work-group's strip is up to 16
// outputs, whose gate rows half of its waves walk and whose up rows the other half (R == 1: each
// wave streams one strip of 16 rows, which is what reaches the memory's rate; four strips per
// wave, as an earlier version had, stayed at 56-58 us on the 7B's matrix where this takes 50-53);
// out has N / 2 columns.
// XL (x through shared memory): with more than one activation row the 16 lanes of a group read
// 16 different rows of x, which no longer fit the L1 cache once M * K * 2 bytes exceed it, and
// every operand load of x becomes a trip to L2 that competes with the weight stream (measured:
// 5.6 TB/s at M = 1, 4.6 at M = 8, 3.7 at M = 16 without it).  With XL the work-group copies
// its M rows of x into shared memory once, coalesced, and reads the operands from there.
// D: how many K steps of weights a wave keeps in flight (a ring of D register sets).  Short
// rows (a few steps per wave) want them all in flight at once, or every step costs a trip to memory.
// RP (the fused query/key/value projection of a decode step, R == 1 and MT == 1): the epilogue rotates
// the query and key heads by the token's position and puts keys and values into their pages, so no
// kernel of its own has to.  The projection's rows are in the pair layout: the two elements that
// frequency j turns are the neighbouring output columns 2j and 2j + 1 of a head, both in one lane.
struct RopeArgs {
    const int* positions;      // [M]
    const float* inv_freq;     // [head_dim / 2]
    const int* token_req;      // [M] request of each row (null: no cache write)
    const int* block_table;    // [requests, bt_stride]
    bf16_t* k_plane;           // [pages, kv_heads, page, head_dim]
    bf16_t* v_plane;           // [pages, kv_heads, head_dim, page]
    int bt_stride, page, q_heads, kv_heads, head_dim;
};

// Four neighbouring columns n .. n + 3 of row m, those below n_end: two pairs (pair layout: one frequency turns a pair; a run of columns ends between pairs or not at all), the query
// and key heads' turned by the row's position `pos`; queries go to out, keys and values to page `page`.
__device__ __forceinline__ void rope_store(const RopeArgs& ra, const f32x4_t& sum, int n, int n_end, int m, int pos, int page, bf16_t* out, int ldo) {
#pragma unroll
    for (int pr = 0; pr < 2; ++pr) {
        const int np = n + 2 * pr;
        if (np + 1 >= n_end) continue;                 // runs hold an even number of columns
        float y1 = sum[2 * pr], y2 = sum[2 * pr + 1];
        const int head = np / ra.head_dim, dd = np - head * ra.head_dim;
        if (head < ra.q_heads + ra.kv_heads) {
            const float angle = (float)pos * ra.inv_freq[dd / 2];
            const float c = cosf(angle), sn = sinf(angle);
            const float t1 = y1 * c - y2 * sn;
            const float t2 = y2 * c + y1 * sn;
            y1 = t1;
            y2 = t2;
        }
        const uint16_t e1 = from_float<bf16_t>(y1).bits, e2 = from_float<bf16_t>(y2).bits;
        const uint32_t both = (uint32_t)e1 | ((uint32_t)e2 << 16);
        if (head < ra.q_heads || !ra.k_plane) {
            *(uint32_t*)(out + (size_t)m * ldo + np) = both;
        } else if (page != 0) {     // page 0 is the sentinel (a padding row's): never written
            const int kvh = (head - ra.q_heads) % ra.kv_heads, off = pos % ra.page;
            const size_t base = ((size_t)page * ra.kv_heads + kvh) * ra.page * ra.head_dim;
            if (head < ra.q_heads + ra.kv_heads) {
                *(uint32_t*)(ra.k_plane + base + (size_t)off * ra.head_dim + dd) = both;
            } else {
                ra.v_plane[base + (size_t)dd * ra.page + off].bits = e1;
                ra.v_plane[base + (size_t)(dd + 1) * ra.page + off].bits = e2;
            }
        }
    }
}

// Eight neighbouring elements as floats, from float or bfloat16 memory and back.
__device__ __forceinline__ void load8(const float* p, float* v) {
    const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ void load8(const bf16_t* p, float* v) {
    const uint4 t = *(const uint4*)p;
    v[0] = __uint_as_float(t.x << 16); v[1] = __uint_as_float(t.x & 0xffff0000u);
    v[2] = __uint_as_float(t.y << 16); v[3] = __uint_as_float(t.y & 0xffff0000u);
    v[4] = __uint_as_float(t.z << 16); v[5] = __uint_as_float(t.z & 0xffff0000u);
    v[6] = __uint_as_float(t.w << 16); v[7] = __uint_as_float(t.w & 0xffff0000u);
}
__device__ __forceinline__ void store8(float* p, const float* v) {
    *(float4*)p = make_float4(v[0], v[1], v[2], v[3]);
    *(float4*)(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}
__device__ __forceinline__ void store8(bf16_t* p, const float* v) {
    uint4 t;
    t.x = (uint32_t)from_float<bf16_t>(v[0]).bits | ((uint32_t)from_float<bf16_t>(v[1]).bits << 16);
    t.y = (uint32_t)from_float<bf16_t>(v[2]).bits | ((uint32_t)from_float<bf16_t>(v[3]).bits << 16);
    t.z = (uint32_t)from_float<bf16_t>(v[4]).bits | ((uint32_t)from_float<bf16_t>(v[5]).bits << 16);
    t.w = (uint32_t)from_float<bf16_t>(v[6]).bits | ((uint32_t)from_float<bf16_t>(v[7]).bits << 16);
    *(uint4*)p = t;
}

// r += the N slabs' eight elements at src, src + stride, ...: all requested, then added in their order.
template <int N>
__device__ __forceinline__ void add_slabs8(const float* src, size_t stride, float (&r)[8]) {
    float p[N][8];
#pragma unroll
    for (int u = 0; u < N; ++u) load8(src + u * stride, p[u]);
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
        for (int v = 0; v < 8; ++v) r[v] += p[u][v];
}

// NF (one row, with XL): x is not read but made here, as the norm of the residual stream would make it:
// r = residual + pending (bfloat16, or float slabs of partial sums), x = r * rsqrt(mean(r^2) + eps) * weight, all
// in 32-bit and rounded once; the first work-group writes r out as the new residual (to another place than it
// is read from: the others may still be reading).  Every work-group does this once for all the strips it
// walks, while its first weights are on their way; the norm's own kernel, a launch and a trip to memory with
// nothing else to do, is not run at all (7B sizes, one row: 4.6 us twice a layer).
struct NormArgs {
    const float* residual;     // [K]
    float* residual_out;       // [K]
    const void* pending;       // bfloat16 [K], or float [parts][part_stride], or null
    const void* weight;        // [K], bfloat16 or float
    size_t part_stride;
    int parts, weight_f32;
    float eps;
    int share, strips, shares;      // TURN: see gemm_skinny_kernel
};

template <int R, int MT, int KS, typename TOut, int SW = 0, bool XL = false, int D = 2, bool RP = false, bool NF = false, bool TURN = false>
__global__ __launch_bounds__(KS * 64) void gemm_skinny_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                              const void* __restrict__ bias, int bias_f32,
                                                              TOut* __restrict__ out, int M, int N, int K, int ldx, int ldo,
                                                              int out_cols, int k_per_split, int rows_per_strip, int rows_per_group,
                                                              RopeArgs ra, NormArgs na, GroupStride gs) {
    static_assert(!NF || (XL && MT == 1), "the fused norm makes x in shared memory, for one row");
    static_assert(!SW || (R == 1 && KS % 2 == 0), "the fused gate deals a work-group's waves to a gate strip and its up strip");
    static_assert(!RP || (R <= 2 && MT == 1 && !SW), "the fused rotation is built for up to 16 rows of x");
    // Split K (k_per_split > 0, a multiple of 64): blockIdx.y owns the columns
    // [y * k_per_split, ...) of x and w and writes its own [M, ldo] slab of partial sums to out
    // (float, no bias); whoever reads them adds the slabs up.
    const int ldw = K;
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
    extern __shared__ __attribute__((aligned(16))) float skinny_lds[];
    float* red = skinny_lds;                                             // KS * R * MT * 256 floats
    bf16_t* xs = (bf16_t*)(skinny_lds + KS * R * MT * 256);             // XL: M rows of K + 8 elements
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, lg = lane >> 4;
    // The outputs (weight rows; with the fused gate, SW, pairs of a gate row and an up row) are dealt to the
    // work-groups in runs of rows_per_group, and a work-group walks its run in strips of rows_per_strip, up to
    // 16 R (0: exactly that; rows_per_group 0: one strip).  A compute unit draws its weights at a rate of its
    // own, about 26 GB/s whatever it shares the chip with, so a product takes as long as its busiest unit: 257
    // strips of 16 rows take as long as 512 (11.2 against 7.9 us for 256, at 3584 columns), and equal shares for
    // all work-groups are worth more than full blocks of 16 rows.  Lanes beyond a strip's last row fetch copies
    // of it and store nothing.  Only with x in shared memory (XL) does a work-group walk more than one strip:
    // x is copied (or made, NF) once for all of them, and the first fetches of the next strip are on their way
    // while the sums of this one are added up.
    // With the fused gate the first KS / 2 waves walk K for the gate rows of the strip's outputs, the others
    // for the up rows of the same outputs (the interleaved matrix holds blocks of 32 gate rows followed by
    // their 32 up rows), and the sums of both meet in shared memory.
    constexpr int KW = SW ? KS / 2 : KS;       // waves along K per strip
    const int kwave = SW ? wave % KW : wave;
    static_assert(!TURN || (NF && !SW && KS == 8), "the rings' order is kept by eight waves along K");
    // The columns that step i of this wave begins at.  TURN: in the order in which gemm_ring_kernel takes them, which begins elsewhere in each of its work-groups (its wave v takes slabs v, v + 4,
    // ... from its start on, for two sums in turn: those are this kernel's waves v and v + 4).
    const int per_wave = K / 256;
    int from = 0;                              // (of the strip at hand)
    auto step_at = [&](int i) {
        if (!TURN) return 64 * (kwave + i * KW);
        const int t = (kwave >> 2) + 2 * i + from;
        return 64 * ((kwave & 3) + 4 * (t < per_wave ? t : t - per_wave));
    };
    const int total = SW ? out_cols : N;
    const int rps = rows_per_strip > 0 ? rows_per_strip : 16 * R;
    const int run_begin = blockIdx.x * ((XL && rows_per_group > 0) ? rows_per_group : rps);
    const int run_end = min(total, run_begin + ((XL && rows_per_group > 0) ? rows_per_group : rps));
    // TURN: the run is na.shares of what gemm_ring_kernel's work-groups have each (na.share outputs), every one of them na.strips strips; the strip's number is then 256 times the share's and its own in it
    auto strip_begin = [&](int i) { return TURN ? run_begin + (i >> 8) * na.share + (i & 255) * rps : run_begin + i * rps; };
    auto strip_end = [&](int i) { return min(TURN ? min(strip_begin(i) + rps, run_begin + ((i >> 8) + 1) * na.share) : run_begin + i * rps + rps, run_end); };
    auto strip_after = [&](int i) { return !TURN || (i & 255) + 1 < na.strips ? i + 1 : (i | 255) + 1; };
    auto turn_to = [&](int i) { if (TURN) from = ring_start(blockIdx.x * na.shares + (i >> 8), per_wave); };
    auto lane_row = [&](int i, int r) {        // the weight row this lane fetches for block r of strip i
        const int o = min(strip_begin(i) + r * 16 + li, strip_end(i) - 1);
        return SW ? (o >> 5) * 64 + (wave / KW) * 32 + (o & 31) : o;
    };
    int strip = 0;
    turn_to(strip);
    int rp_pos = 0, rp_page = 0;               // RP: this lane's row (li), fetched now, used in the epilogue
    if (RP) {
        const int row = min(li, M - 1);
        rp_pos = ra.positions[row];
        if (ra.k_plane) rp_page = ra.block_table[(size_t)ra.token_req[row] * ra.bt_stride + rp_pos / ra.page];
    }

    const bf16_t* wrow[R];
    const bf16_t* xrow[MT];
    int xoff[MT];
#pragma unroll
    for (int r = 0; r < R; ++r) wrow[r] = w + (size_t)lane_row(strip, r) * ldw;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        xrow[t] = x + (size_t)min(t * 16 + li, M - 1) * ldx;
        xoff[t] = min(t * 16 + li, M - 1) * (K + 8);
    }
#define SK_LOADB(t, k) (XL ? *(const uint4*)(&xs[xoff[t] + (k)]) : *(const uint4*)(xrow[t] + (k)))

    f32x4_t acc[R][MT];
    const int full = K / 64;                   // steps that lie wholly inside K
    // this wave's steps are s = kwave + i * KW, i = 0 .. mine - 1; slot d of the ring holds step i = d (mod D)
    const int mine = full > kwave ? (full - kwave + KW - 1) / KW : 0;
    Frag16 wa0[D][R], wa1[D][R], wb0[D][MT], wb1[D][MT];
#define SK_ISSUE(d, i)                                                                              \
    {                                                                                               \
        const int k_ = step_at(i) + SK_KOFF(lg);                                                    \
        _Pragma("unroll") for (int r = 0; r < R; ++r) {                                             \
            wa0[d][r].u = SK_LOAD(wrow[r] + k_);                                                    \
            wa1[d][r].u = SK_LOAD(wrow[r] + k_ + SK_SECOND);                                        \
        }                                                                                           \
        if (!XL) {                                                                                  \
            _Pragma("unroll") for (int t = 0; t < MT; ++t) {                                        \
                wb0[d][t].u = SK_LOAD(xrow[t] + k_);                                                \
                wb1[d][t].u = SK_LOAD(xrow[t] + k_ + SK_SECOND);                                    \
            }                                                                                       \
        }                                                                                           \
    }
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (d < mine) SK_ISSUE(d, d)
    if (NF) {                                  // the weights are on their way while x is made
        // a thread owns up to two pieces of eight elements (the host checked K <= 16 * threads)
        const int pieces = K / 8;
        float r[2][8];
        float ss = 0.f;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int i = min((int)threadIdx.x + c * KS * 64, pieces - 1) * 8;
            load8(na.residual + i, r[c]);
            if (na.pending && na.parts == 0) {
                float p[8];
                load8((const bf16_t*)na.pending + i, p);
#pragma unroll
                for (int v = 0; v < 8; ++v) r[c][v] += p[v];
            }
            const float* slab = (const float*)na.pending + i;
            if constexpr (RP) {
                // The query/key/value projection follows the down projection, whose K is split many ways: four slabs
                // at a time, all requested before the first is added, in their order (one after the other, the eight
                // slabs of the 7B's down projection were eight trips to memory before the first weight was used); the
                // last two or three are a group as well.
                int q = 0;
                for (; q + 4 <= na.parts; q += 4) add_slabs8<4>(slab + q * na.part_stride, na.part_stride, r[c]);
                if (na.parts - q == 3) add_slabs8<3>(slab + q * na.part_stride, na.part_stride, r[c]);
                else if (na.parts - q == 2) add_slabs8<2>(slab + q * na.part_stride, na.part_stride, r[c]);
                else if (na.parts - q == 1) add_slabs8<1>(slab + q * na.part_stride, na.part_stride, r[c]);
            } else {
                // (the fused gate follows the output projection, one slab or few: the registers of a group would cost
                // its work-groups of sixteen waves the second one on a compute unit)
                for (int q = 0; q < na.parts; ++q) {
                    float p[8];
                    load8(slab + q * na.part_stride, p);
#pragma unroll
                    for (int v = 0; v < 8; ++v) r[c][v] += p[v];
                }
            }
            if ((int)threadIdx.x + c * KS * 64 < pieces) {
#pragma unroll
                for (int v = 0; v < 8; ++v) ss += r[c][v] * r[c][v];
            }
        }
        ss = wave_sum(ss);
        float* sums = red;                            // free until the first strip's sums
        if (lane == 0) sums[wave] = ss;
        lds_barrier();
        float total = 0.f;
        for (int wv = 0; wv < KS; ++wv) total += sums[wv];
        const float inv = rsqrtf(total / (float)K + na.eps);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int pc = (int)threadIdx.x + c * KS * 64;
            if (pc < pieces) {
                float g[8];
                if (na.weight_f32) load8((const float*)na.weight + pc * 8, g);
                else load8((const bf16_t*)na.weight + pc * 8, g);
                float o[8];
#pragma unroll
                for (int v = 0; v < 8; ++v) o[v] = r[c][v] * inv * g[v];
                store8(xs + pc * 8, o);
                if (blockIdx.x == 0 && blockIdx.y == 0) {
                    store8(na.residual_out + pc * 8, r[c]);
                }
            }
        }
        lds_barrier();
    } else if (XL) {                           // the weights are on their way while x is copied
        const int pieces = K / 8;                     // 16-byte pieces per row
        for (int i = threadIdx.x; i < M * pieces; i += KS * 64) {
            const int row = i / pieces, pc = i % pieces;
            *(uint4*)(&xs[row * (K + 8) + pc * 8]) = *(const uint4*)(x + (size_t)row * ldx + pc * 8);
        }
        lds_barrier();
    }
    while (true) {
        const int n0 = strip_begin(strip);     // first output column of the strip
        const int n_end = strip_end(strip);    // ... and the one after its last
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[r][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        for (int i = 0; i < mine; i += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                if (i + d < mine) {
                    if (XL) {
                        const int k = step_at(i + d) + SK_KOFF(lg);
#pragma unroll
                        for (int t = 0; t < MT; ++t) {
                            wb0[d][t].u = *(const uint4*)(&xs[xoff[t] + k]);
                            wb1[d][t].u = *(const uint4*)(&xs[xoff[t] + k + SK_SECOND]);
                        }
                    }
#pragma unroll
                    for (int r = 0; r < R; ++r)
#pragma unroll
                        for (int t = 0; t < MT; ++t) {
                            acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa0[d][r].v, wb0[d][t].v, acc[r][t], 0, 0, 0);
                            acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa1[d][r].v, wb1[d][t].v, acc[r][t], 0, 0, 0);
                        }
                    if (i + d + D < mine) SK_ISSUE(d, i + d + D)
                }
            }
        }
        // the tail step (K % 64 != 0) belongs to the wave whose turn it is; pieces beyond K count as zero
        if ((K & 63) && (full % KW) == kwave) {
            Frag16 a0[R], a1[R], b0[MT], b1[MT];
            const int k = 64 * full + SK_KOFF(lg);
            const bool v0 = k + 8 <= K, v1 = k + SK_SECOND + 8 <= K;
            // (fetched from a clamped address and cleared afterwards: a fetch under a condition makes the
            // compiler route it through scratch memory, which every launch of the kernel then sets up)
            const int k0 = min(k, K - 8), k1 = min(k + SK_SECOND, K - 8);
            auto keep = [](uint4 v, bool ok) {
                v.x = ok ? v.x : 0u;
                v.y = ok ? v.y : 0u;
                v.z = ok ? v.z : 0u;
                v.w = ok ? v.w : 0u;
                return v;
            };
#pragma unroll
            for (int r = 0; r < R; ++r) {
                a0[r].u = keep(*(const uint4*)(wrow[r] + k0), v0);
                a1[r].u = keep(*(const uint4*)(wrow[r] + k1), v1);
            }
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                b0[t].u = keep(SK_LOADB(t, k0), v0);
                b1[t].u = keep(SK_LOADB(t, k1), v1);
            }
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[r].v, b0[t].v, acc[r][t], 0, 0, 0);
                    acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[r].v, b1[t].v, acc[r][t], 0, 0, 0);
                }
        }
        const int next = strip_after(strip);
        const bool more = XL && strip_begin(next) < run_end;        // without the copy of x: one strip per work-group
        if (more) {                            // the next strip's first steps, before this strip's sums
#pragma unroll
            for (int r = 0; r < R; ++r) wrow[r] = w + (size_t)lane_row(next, r) * ldw;
            turn_to(next);
#pragma unroll
            for (int d = 0; d < D; ++d)
                if (d < mine) SK_ISSUE(d, d)
        }

        // D[i][j]: lane holds i = 4 * (lane / 16) + v (weight row), j = lane % 16 (activation row)
        if (KS > 1) {
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    float* dst = red + ((size_t)(wave * R * MT + r * MT + t) * 64 + lane) * 4;
                    *(f32x4_t*)dst = acc[r][t];
                }
            lds_barrier();
        }
        if (SW) {
            for (int t = wave; t < MT; t += KS) {
                f32x4_t gs = f32x4_t{0.f, 0.f, 0.f, 0.f}, us = gs;
#pragma unroll
                for (int wv = 0; wv < KW; ++wv) {
                    gs += *(const f32x4_t*)(red + ((size_t)(wv * MT + t) * 64 + lane) * 4);
                    us += *(const f32x4_t*)(red + ((size_t)((KW + wv) * MT + t) * 64 + lane) * 4);
                }
                const int m = t * 16 + li;
                const int col = n0 + 4 * lg;
                if (m < M) {
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (col + v < n_end) out[(size_t)m * ldo + col + v] = from_float<TOut>(gate_mul<SW>(gs[v], us[v]));
                }
            }
        } else {
            for (int tile = wave; tile < R * MT; tile += KS) {
                const int r = tile / MT, t = tile % MT;
                f32x4_t sum;
                if (KS > 1) {
                    sum = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int wv = 0; wv < KS; ++wv) sum += *(const f32x4_t*)(red + ((size_t)(wv * R * MT + tile) * 64 + lane) * 4);
                } else {
                    sum = acc[0][0];
#pragma unroll
                    for (int rr = 0; rr < R; ++rr)
#pragma unroll
                        for (int tt = 0; tt < MT; ++tt)
                            if (rr == r && tt == t) sum = acc[rr][tt];
                }
                const int m = t * 16 + li;
                const int n = n0 + r * 16 + 4 * lg;
                if (RP) {
                    if (bias) {
#pragma unroll
                        for (int v = 0; v < 4; ++v) sum[v] += load_vec(bias, bias_f32, min(n + v, N - 1));
                    }
                    if (m < M) rope_store(ra, sum, n, n_end, m, rp_pos, rp_page, (bf16_t*)out, ldo);
                    continue;
                }
                if (m < M) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        if (n + v < n_end) {
                            float val = sum[v];
                            if (bias) val += load_vec(bias, bias_f32, n + v);
                            out[(size_t)m * ldo + n + v] = from_float<TOut>(val);
                        }
                    }
                }
            }
        }
        if (!more) break;
        strip = next;
        if (KS > 1) lds_barrier();             // the sums are read until here; the next strip's overwrite them
    }
#undef SK_ISSUE
}

#define SKINNY_XL_MAX_BYTES (60 * 1024)      // x may take this much shared memory: with the reduction buffer two
                                             // work-groups still fit the 160 KB of a compute unit

// How the outputs of a product are dealt out: work-groups, the outputs of each (its run) and of a strip.
struct StripPlan {
    int groups, per_group, per_strip;
};

// A run of outputs in equal strips of at most `cap` (a multiple of 16; `even`: of an even number).
static int equal_strips(int run, int cap, bool even) {
    const int count = (run + cap - 1) / cap, rows = (run + count - 1) / count;
    return even ? rows + (rows & 1) : rows;
}

// Equal runs for up to `most` work-groups, each walked in equal strips of at most `cap` outputs (a multiple of
// 16); `even` keeps both numbers even (the fused rotation turns pairs of neighbouring outputs).
static StripPlan plan_strips(int total, int most, int cap, bool even) {
    StripPlan p;
    p.per_group = (total + most - 1) / most;
    if (p.per_group < 4) p.per_group = 4;                     // a strip of fewer rows wastes most of its fetches
    if (even) p.per_group += p.per_group & 1;
    p.per_strip = equal_strips(p.per_group, cap, even);
    p.groups = (total + p.per_group - 1) / p.per_group;
    return p;
}

// rows_per_strip > 0: one strip of that many outputs per work-group, whatever else holds.
template <int R, int MT, int KS, typename TOut, int SW, int D>
static void launch_skinny_d(const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int N, int K,
                            int ldx, int ldo, int out_cols, hipStream_t stream, int rows_per_strip = 0, Groups gr = Groups{}) {
    const int total = SW ? out_cols : N;
    const int rps = rows_per_strip > 0 ? rows_per_strip : 16 * R;
    dim3 grid((total + rps - 1) / rps, 1, gr.count), block(KS * 64);
    const size_t red_bytes = (size_t)KS * R * MT * 1024;
    const size_t x_bytes = (size_t)M * (K + 8) * 2;
    // More than one row of x: two work-groups per compute unit copy x into shared memory once and walk
    // their runs of outputs (each strip's own copy took longer than it saved: 87 against 64 us on the
    // fused gate/up product at M = 8 with four waves).
    if (M > 1 && red_bytes + x_bytes <= 156 * 1024) {
        auto kernel = gemm_skinny_kernel<R, MT, KS, TOut, SW, true, D>;
        static hipError_t allowed = allow_lds(kernel, 156 * 1024);
        if (allowed == hipSuccess) {
            const int most = (x_bytes <= SKINNY_XL_MAX_BYTES ? 2 * TL_COMPUTE_UNITS : TL_COMPUTE_UNITS) / gr.count;      // a larger x leaves room for one work-group only
            StripPlan p = plan_strips(total, most > 0 ? most : 1, 16 * R, false);
            if (rows_per_strip > 0) p = StripPlan{(int)grid.x, rps, rps};
            kernel<<<dim3(p.groups, 1, gr.count), block, red_bytes + x_bytes, stream>>>((const bf16_t*)x, (const bf16_t*)w, bias, bias_f32, (TOut*)out, M, N, K, ldx, ldo,
                                                                           out_cols, 0, p.per_strip, p.per_group, RopeArgs{}, NormArgs{}, gr.stride);
            return;
        }
    }
    gemm_skinny_kernel<R, MT, KS, TOut, SW, false, D><<<grid, block, red_bytes, stream>>>((const bf16_t*)x, (const bf16_t*)w, bias, bias_f32, (TOut*)out, M, N, K, ldx, ldo,
                                                                                          out_cols, 0, rps, 0, RopeArgs{}, NormArgs{}, gr.stride);
}

// A wave with many K steps ahead of it (a long K: the down projection) keeps as many in flight as
// its registers hold; with a few steps (K of a hidden size) two are as good and start sooner
// (measured at 3584 x 18944, one row: 33 -> 28 us with eight in flight; at 4608 x 3584: 11 -> 12.6 us).
template <int R, int MT, int KS, typename TOut, int SW>
static void launch_skinny_t(const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int N, int K,
                            int ldx, int ldo, int out_cols, hipStream_t stream, int rows_per_strip = 0, Groups gr = Groups{}) {
    constexpr int deep = skinny_depth<R, MT, KS>();
    if (deep > 2 && K / 64 / KS >= 16)
        launch_skinny_d<R, MT, KS, TOut, SW, deep>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_cols, stream, rows_per_strip, gr);
    else
        launch_skinny_d<R, MT, KS, TOut, SW, 2>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_cols, stream, rows_per_strip, gr);
}

template <int R, int MT, int KS>
static void launch_skinny(const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int N, int K,
                          int ldx, int ldo, int out_f32, hipStream_t stream, int rows_per_strip = 0, Groups gr = Groups{}) {
    if (out_f32) launch_skinny_t<R, MT, KS, float, false>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, 0, stream, rows_per_strip, gr);
    else launch_skinny_t<R, MT, KS, bf16_t, false>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, 0, stream, rows_per_strip, gr);
}

// Rows a strip gets so that a matrix of N rows is dealt to the compute units in equal shares, one strip to
// each (0: the plain strips of 16 R rows are as good; *blocks: how many blocks of 16 rows a strip then has, 1 or
// 2).  A compute unit draws its weights at a rate of its own, about 26 GB/s whatever shares it with, and the strips
// beyond one per unit run when the others are done, nearly alone, at the latency of every fetch: at 3584 columns 256 strips of 16 rows take 7.9 us, 257 take 11.2, 288 (the
// 7B's query/key/value matrix) 11.9 and 512 take 13.4.  The number is even (the fused rotation turns pairs).
static int balanced_rows(int N, int* blocks) {
    *blocks = 1;
    if (N < 4 * TL_COMPUTE_UNITS || N > 32 * TL_COMPUTE_UNITS) return 0;      // a few rows a unit, or more than two blocks
    if (N % (16 * TL_COMPUTE_UNITS) == 0) return 0;                               // whole blocks already come out even
    int rows = (N + TL_COMPUTE_UNITS - 1) / TL_COMPUTE_UNITS;
    rows += rows & 1;
    *blocks = rows > 16 ? 2 : 1;
    return rows;
}

template <int MT>
static void pick_skinny(const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int N, int K,
                        int ldx, int ldo, int out_f32, hipStream_t stream, Groups gr = Groups{}) {
    // Measured on MI355X at Qwen2.5-7B sizes (weights streamed from HBM, M = 8 and 64; K a multiple of 64, which but for one row against many columns the rings take by now):
    // with up to 32 rows one strip of 16 weight rows per work-group is best throughout, with
    // 16 waves along K for wide matrices (gate_up, LM head: 4.7-5.0 TB/s) and 8 for narrow
    // ones (qkv, o, down); with 64 rows the x operand weighs more and several strips per wave
    // share each x load.
    const int strips = (N + 15) / 16 * gr.count;
    if (MT == 1 && gr.count == 1) {
        int blocks = 1;
        const int rows = balanced_rows(N, &blocks);
        if (rows > 0 && blocks == 1) return launch_skinny<1, 1, 8>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_f32, stream, rows);
        if (rows > 0) return launch_skinny<2, 1, 8>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_f32, stream, rows);
    }
    if (MT <= 2) {
        if (strips >= 1024) launch_skinny<1, MT, 16>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_f32, stream, 0, gr);
        else launch_skinny<1, MT, 8>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_f32, stream, 0, gr);
    } else {
        if (strips >= 2048) launch_skinny<4, MT, 4>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_f32, stream, 0, gr);
        else if (strips >= 1024) launch_skinny<2, MT, 2>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_f32, stream, 0, gr);
        else launch_skinny<1, MT, 8>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_f32, stream, 0, gr);
    }
}

// ------------------------------------------------------------------ few rows through rings in shared memory (K a multiple of 64)
// See row_ring.h.  Work-group (i, y, z): outputs i * rps .. of product z (gs), or the y-th range of K of a product split over K (k_per_split columns each, a
// slab [M, ldo] of partial sums each).  SW: the gate's activation as in gemm_skinny_kernel (out_cols outputs, gate and up rows interleaved in blocks of 32); END: what becomes of the
// sums: END_ROTATE its rotation and cache write, END_TOKEN an activation and the product with the row's token's own numbers (16 rows, 256 x 2048: 5.6 us in two launches, 4.4 in one);
// END_BESIDE: as END_STORE, and behind the products of gs comes one more (blockIdx.z == be.z), of other columns and into float, eight of them to a work-group: it shares its compute
// unit with another one (16 rows, 4 x 2048 x 2048 and 64 x 2048: 12.9 us in two launches, 10.7 in one, 11.8 with as many columns to a work-group as the others have).
#define END_STORE 0
#define END_ROTATE 1
#define END_TOKEN 2
#define END_BESIDE 3
struct Beside {
    const bf16_t *x, *w;      // rows of x as far apart as the others'
    float* out;               // [M, N]
    int N, z;
};
struct TokenRow {
    const int* ids;
    const bf16_t* table;      // row ids[m] holds N numbers; rows ld apart; what is no row leaves its outputs as they are
    int ld, vocab, act;
};
template <int WJ, int XH, typename TOut, int SW = 0, int END = END_STORE, typename T = bf16_t>
__global__ __launch_bounds__((64 * ring_waves<WJ, T>())) void gemm_ring_kernel(const T* __restrict__ x, const T* __restrict__ w, const void* __restrict__ bias, int bias_f32,
                                                        TOut* __restrict__ out, int M, int N, int K, int ldx, int ldo, int out_cols, int k_per_split, int rps,
                                                        RopeArgs ra, TokenRow tk, Beside be, GroupStride gs, F32Pairs pa) {
    constexpr bool RP = END == END_ROTATE, TK = END == END_TOKEN, BE = END == END_BESIDE;
    constexpr bool PAIRS = sizeof(T) == 4 && (SW || RP);      // float: rows by pairs (F32Pairs); out_cols counts them
    constexpr int HALVES = SW || PAIRS ? 2 : 1;
    using S = RingShape<WJ, XH, HALVES, T>;
    static_assert(END == END_STORE || END == END_BESIDE || (!SW && S::MT == 1 && (sizeof(TOut) == 2 || PAIRS)), "the rotation and the tokens' rows are built for up to 16 rows");
    extern __shared__ __attribute__((aligned(16))) char ring[];
    const int ldw = K;
    const bool beside = BE && (int)blockIdx.z == be.z;
    if (BE) {
        if (beside) {
            x = (const T*)be.x;
            w = (const T*)be.w;
            N = be.N;
            rps = min(rps, 8);
        }
        if ((int)blockIdx.x * rps >= N) return;        // (the whole work-group: the grid is as wide as the widest product)
    }
    if (!beside) {
        x += blockIdx.z * gs.x;
        w += blockIdx.z * gs.w;
        out += blockIdx.z * gs.out;
    }
    if (k_per_split > 0) {
        const int kb = blockIdx.y * k_per_split;
        x += kb;
        w += kb;
        out += (size_t)blockIdx.y * M * ldo;
        K = min(K - kb, k_per_split);
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 15, kg = lane >> 4;
    const int n0 = blockIdx.x * rps, n_end = min(HALVES == 2 ? out_cols : N, n0 + rps);
    // (the waves that turn and write: their rows' positions and pages ahead of the weights, so that no wait for them lies behind the ring's)
    int rp_pos = 0, rp_page = 0;
    float2 rp_turn[4] = {};
    if (PAIRS && RP && wave < S::SH) {
        const int row = min(li, M - 1);
        rp_pos = pa.positions[row];
        if (pa.k_plane) rp_page = pa.block_table[(size_t)pa.token_req[row] * pa.bt_stride + rp_pos / pa.page];
#pragma unroll
        for (int v = 0; v < 4; ++v) rp_turn[v] = f32_turn(pa, n0 + 16 * wave + 4 * kg + v, rp_pos);
    } else if (RP && !PAIRS && wave < S::STRIPS) {
        const int row = min(li, M - 1);
        rp_pos = ra.positions[row];
        if (ra.k_plane) rp_page = ra.block_table[(size_t)ra.token_req[row] * ra.bt_stride + rp_pos / ra.page];
    }
    const int tk_id = TK ? tk.ids[min(li, M - 1)] : 0;
    // the matrix's row of an output's gate (or of the output itself); its up row lies 32 further on, a pair's second row a span
    auto row_of = [&](int o) { return PAIRS ? pa.row(o) : SW ? (o >> 5) * 64 + (o & 31) : o; };
    const int apart = PAIRS ? pa.span : 32;
    unsigned woff[WJ], xoff[XH];
#pragma unroll
    for (int j = 0; j < WJ; ++j) {
        const int r = 8 * j + lane / 8, c = (lane % 8) ^ ((r >> 1) & 7), half = r / S::HR;
        woff[j] = (unsigned)(row_of(min(n0 + r - half * S::HR, n_end - 1)) - row_of(n0) + apart * half) * (unsigned)ldw * (unsigned)sizeof(T) + c * 16;
    }
#pragma unroll
    for (int j = 0; j < XH; ++j) {
        const int r = 8 * (WJ + j) + lane / 8, c = (lane % 8) ^ ((r >> 1) & 7);
        xoff[j] = (unsigned)(min(r - 8 * WJ, M - 1) * ldx) * (unsigned)sizeof(T) + c * 16;
    }
    ring_products<WJ, XH, HALVES>(w + (size_t)row_of(n0) * ldw, woff, x, xoff, K / (128 / (int)sizeof(T)), ring, wave, ring_spread<T>(ldw));
    const bool quads = ldo % 4 == 0 && n0 % 4 == 0 && ((uintptr_t)out % (4 * sizeof(TOut))) == 0;
    for (int q = wave; q < S::SH * S::MT; q += S::NW) {
        const int s = q / S::MT, t = q % S::MT, m = 16 * t + li, n = n0 + 16 * s + 4 * kg;
        const bool known = !TK || (tk_id >= 0 && tk_id < tk.vocab);
        float own[4];
        if constexpr (TK) {
#pragma unroll
            for (int v = 0; v < 4; ++v) own[v] = known ? to_float(tk.table[(size_t)tk_id * tk.ld + min(n + v, N - 1)]) : 0.f;
        }
        f32x4_t sum = ring_sum<WJ, XH, HALVES, T>(ring, s, t);
        if constexpr (PAIRS) {
            const f32x4_t up = ring_sum<WJ, XH, HALVES, T>(ring, S::SH + s, t);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                float a = sum[v], b = up[v];
                if (SW) {
                    sum[v] = f32_gate(pa.act, a, b);
                } else if (m < M && n + v < n_end) {
                    if (bias) { a += load_vec(bias, bias_f32, pa.row(n + v)); b += load_vec(bias, bias_f32, pa.row(n + v) + pa.span); }
                    f32_turn_store(pa, n + v, a, b, rp_turn[v], m, rp_pos, rp_page, (float*)out, ldo);
                }
            }
            if (RP) continue;
        } else if constexpr (SW) {
            const f32x4_t up = ring_sum<WJ, XH, HALVES, T>(ring, S::SH + s, t);
#pragma unroll
            for (int v = 0; v < 4; ++v) sum[v] = gate_mul<SW>(sum[v], up[v]);
        } else if (bias) {
#pragma unroll
            for (int v = 0; v < 4; ++v) sum[v] += load_vec(bias, bias_f32, min(n + v, N - 1));
        }
        if (m >= M || !known) continue;
        if constexpr (TK) {
#pragma unroll
            for (int v = 0; v < 4; ++v) sum[v] = activate(sum[v], tk.act) * own[v];
        }
        if (beside) {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (n + v < n_end) be.out[(size_t)m * be.N + n + v] = sum[v];
            continue;
        }
        if constexpr (RP && !PAIRS) {
            rope_store(ra, sum, n, n_end, m, rp_pos, rp_page, (bf16_t*)out, ldo);
        } else if (quads && n + 3 < n_end) {
            store4(out + (size_t)m * ldo + n, make_float4(sum[0], sum[1], sum[2], sum[3]));
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (n + v < n_end) out[(size_t)m * ldo + n + v] = from_float<TOut>(sum[v]);
        }
    }
}

// What the rings take: whole slabs, 16-byte aligned rows, offsets inside a work-group's rows (of the interleaved matrix 128 apart at most) that fit 32 bits.
static bool ring_fits(const void* x, const void* w, int M, int K, int ldx) {
    return M > 0 && M <= 64 && K % 64 == 0 && ldx % 8 == 0 && K < (1 << 23) && ldx < (1 << 23) && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0;
}

// The same in 32 bits: slabs of 32 columns, up to 16 rows.
static bool ring_fits_f32(const void* x, const void* w, int M, int K, int ldx) {
    return M > 0 && M <= 16 && K % 32 == 0 && ldx % 4 == 0 && K < (1 << 22) && ldx < (1 << 22) && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0;
}

// And where they are taken, against the multiply-add kernel (up to 8 rows) and the matrix-core kernel (above) that fetch into registers behind a copy of x and begin every chunk of it with an empty
// pipe (us, those / the rings, weights from memory): 4 rows 4608 x 3584 17.8 / 14.9, 37888 x 3584 109 / 94, 3584 x 18944 61 / 47.6, 152064 x 3584 391 / 360; 8 rows 23 / 15.4, 122 / 95, 87 / 49,
// 454 / 366; 16 rows 25 / 15.7, 131 / 100, 112 / 54, 482 / 374, 512 x 512 4.3 / 3.2; 2048 x 2048 4 rows 8.0 / 6.6, 8 rows 12.4 / 6.7.  Narrow matrices want more work-groups than
// these have (4 rows, 256 x 2048 5.2 / 5.5, 64 x 4096 7.5 / 8.3).
// A ring takes as long for one row as for eight, the multiply-adds do not: one and two rows go to the rings where these are ahead of both, deep matrices, deeper ones where the rows lie multiples of 4 KB
// apart, and neither wide ones nor small ones, which come out of a cache and want their one trip short (one row, 1024 x 1024 3.0 / 4.3, 2048 x 2048 6.0 / 6.6, out of a cache 3.9 / 5.9, 8192 x 1024 8.1 / 9.4, 32768 x 1024
// 23.4 / 28.5, 22016 x 4096 62 / 66, 37888 x 3584 89 / 93, 3584 x 3584 11.7 / 11.4, 4608 x 3584 15.2 / 13.7, 4096 x 8192 30.0 / 26.2, 8192 x 8192 53 / 49; two rows, 1024 x 1024 3.5 / 4.3, 4096 x 3584 0.86, 2560 x 2560
// 0.85, 7168 x 4096 1.18, 6144 x 5120 0.93 of the multiply-adds' time; 16 widths by 18 depths measured).  Whole passes of one and two requests of fifteen models (ms, the
// rings from 1024 x 1024 on / never / by this rule): one request, width 5120 26.0 / 25.1 / 24.8, 3584 14.6 / 14.5 / 14.4, 4096 12.2 / 12.1 / 11.8, 2048 6.20 / 5.96 / 5.93; two, 5120 28.1 / 27.6 / 27.1, 3584
// 15.6 / 15.7 / 15.4, 4096 13.1 / 13.3 / 12.8, 2048 6.24 / 6.35 / 6.12; nowhere behind either by more than two runs differ.
// The sums' error against 64 bits (relative): K 2048 1.2e-7 / 1.0e-7, 3584 1.5e-7 / 1.1e-7, 18944 3.1e-7 / 1.8e-7, above 8 rows
// 3.8e-7 / 1.1e-7; at 512 columns up to 8 rows 0.87e-7 / 0.9e-7, and so short sums stay where they are.
static bool ring_pays_f32(int M, int N, int K) {
    if (M > 2) return M > 8 || (K >= 1024 && N >= 1024);
    const bool apart = K % 1024 == 0;
    return (long)N * K >= 9000000 && (N <= 10240 || K >= 8192) && (M == 1 ? N >= 2048 && K >= (apart ? 8192 : 3584) : N >= 1536 && K >= (apart ? 5120 : 2560));
}
// Which kernel a 32-bit product of up to 16 rows gets whose operands are aligned, by its number in tl_gemm_f32_variant: 9 the rings, 2 multiply-adds, 3 the matrix cores behind a copy of x.  The
// last two part at 8 rows, where a row more costs a multiply-add a weight or nothing (the four products of a 7B layer, us, 2 / 3: 4 rows 216 / 241, 8 rows 274 / 265, 16 rows 425 / 300).
static int f32_few_rows_kernel(int M, int N, int K) { return K % 32 == 0 && ring_pays_f32(M, N, K) ? 9 : M <= 8 ? 2 : 3; }
extern "C" int tl_gemm_f32_few_rows_choice(int M, int N, int K) { return f32_few_rows_kernel(M, N, K); }

// Where a product of up to 64 rows goes through the rings, K a multiple of 64: measured against what it took before them, the tiles or the few-rows kernel that fetches into registers, over a grid
// of widths and depths (us, the other / this).
//   Up to 16 rows up to 32768 columns, 2 to 8 rows any number: 12 rows, 152064 x 3584 190 / 194, 8 rows 197 / 187, 1 row 179 / 187, 2 rows 151936 x 896 53 / 50.
//   17 to 32 rows up to 24576, deep ones up to 32768 (32 rows: 24576 x 1024 13.8 / 11.9, 28672 x 256 6.1 / 7.6, 27648 x 1024 14.3 / 15.9, x 2048 28.4 / 25.4).
//   33 to 64 rows fetch as much of x as of the weights, and the tiles' work-groups share it: up to 8192 columns (64 rows, 2048 x 2048 8.5 / 6.0, 8192 x 1024 8.2 / 6.7, x 256 4.4 / 4.2), up to 24576
//   where K is deep (18432 x 4096 48 / 39, 24576 x 2048 28.5 / 25.4, 16384 x 1024 9.5 / 10.6, 24576 x 256 6.4 / 8.2), with rows of weights multiples of 4 KB apart, whose order the rings turn,
//   up to 32768 (30000 x 4096 55.6 / 54.0, x 5120 64 / 72).
static bool ring_pays(int M, long columns, int K) {
    if (M <= 16) return columns <= 32768 || (M >= 2 && M <= 8);
    if (M <= 32) return columns <= 24576 || (columns <= 32768 && K >= 2048);
    return M <= 64 && (columns <= 8192 || (K >= 2048 && (columns <= 24576 || (columns <= 32768 && K % 2048 == 0))));
}

// The same for a fused gate, `outputs` of which there are (us, the other / this): up to 16 rows but for wide and shallow ones, where the few-rows kernel's work-groups walk many strips each (8 rows,
// 20480 outputs, K 256 7.5 / 8.8, 768 14.1 / 14.8, 1536 25.7 / 23.7; one row, K 768 15.4 / 14.6); 17 to 32 rows up to 12288 outputs (32 rows, 11264 x 4096 46 / 34, 18944 x 3584 50 / 52); 33 to 64
// rows up to 8192, deep ones up to 12288 (64 rows: 8192 x 512 9.1 / 7.2, 11264 x 4096 47 / 44, x 1024 14.8 / 16.5, 12288 x 256 7.2 / 9.4).
static bool ring_pays_gated(int M, int outputs, int K) {
    if (M <= 16) return M == 1 || outputs <= 16384 || K >= 1024;
    return M <= 64 && (outputs <= (M <= 32 ? 12288 : 8192) || (outputs <= 12288 && K >= 2048));
}

struct RingCall {
    const void *x, *w, *bias;
    int bias_f32;
    void* out;
    int M, N, K, ldx, ldo, out_cols;       // out_cols > 0: the fused gate's outputs
    int parts = 1, k_per = 0;
    Groups gr = Groups{};
    RopeArgs ra = RopeArgs{};
    TokenRow tk = TokenRow{};
    Beside be = Beside{};
    F32Pairs pa = F32Pairs{};
};

template <int WJ, int XH, typename TOut, int SW, int END, typename T>
static int launch_ring_t(const RingCall& c, int rows, hipStream_t stream) {
    constexpr int HALVES = SW || (END == END_ROTATE && sizeof(T) == 4) ? 2 : 1;
    using S = RingShape<WJ, XH, HALVES, T>;
    auto kernel = gemm_ring_kernel<WJ, XH, TOut, SW, END, T>;
    static hipError_t allowed = allow_lds(kernel, S::LDS);
    TL_REQUIRE(allowed == hipSuccess, "gemm_ring: cannot get %zu bytes of shared memory", S::LDS);
    const int total = HALVES == 2 ? c.out_cols : c.N, least = min(rows, 8), wide = max((total + rows - 1) / rows, (c.be.N + least - 1) / least);      // (be.N: 0 without a product beside)
    kernel<<<dim3(wide, c.parts, c.gr.count + (END == END_BESIDE)), 64 * S::NW, S::LDS, stream>>>((const T*)c.x, (const T*)c.w, c.bias, c.bias_f32, (TOut*)c.out, c.M, c.N, c.K,
                                                                                      c.ldx, c.ldo, c.out_cols, c.k_per, rows, c.ra, c.tk, c.be, c.gr.stride, c.pa);
    TL_CHECK_LAUNCH("gemm_ring");
    return TL_OK;
}

template <int XH, typename TOut, int SW, int END, typename T>
static int launch_ring_x(const RingCall& c, RingPlan p, hipStream_t stream) {
    switch (p.wj) {
    case 2: return launch_ring_t<2, XH, TOut, SW, END, T>(c, p.rows, stream);
    case 4: return launch_ring_t<4, XH, TOut, SW, END, T>(c, p.rows, stream);
    case 6: return launch_ring_t<6, XH, TOut, SW, END, T>(c, p.rows, stream);
    case 8: return launch_ring_t<8, XH, TOut, SW, END, T>(c, p.rows, stream);
    }
    if constexpr (!SW || sizeof(T) == 4) {
        if (p.wj == 3) return launch_ring_t<3, XH, TOut, SW, END, T>(c, p.rows, stream);
    }
    if constexpr (!SW && !(END == END_ROTATE && sizeof(T) == 4)) {
        if (p.wj == 1) return launch_ring_t<1, XH, TOut, SW, END, T>(c, p.rows, stream);
    }
    TL_REQUIRE(false, "gemm_ring: no shape of %d requests", p.wj);
}

// `p.wj` 0: the plan is made here.
template <typename TOut, int SW, int END, typename T = bf16_t>
static int launch_ring(const RingCall& c, hipStream_t stream, RingPlan p = RingPlan{0, 0}) {
    constexpr bool pairs = sizeof(T) == 4 && (SW || END == END_ROTATE);
    if (p.wj == 0) p = plan_ring(SW || pairs ? c.out_cols : c.N, c.M, SW || pairs ? 2 : 1, TL_COMPUTE_UNITS / (c.parts * c.gr.count), END == END_ROTATE && !pairs, ring_spread<T>(c.K), c.parts > 1, pairs);
    if (c.M <= 8) return launch_ring_x<1, TOut, SW, END, T>(c, p, stream);
    if (c.M <= 16) return launch_ring_x<2, TOut, SW, END, T>(c, p, stream);
    if constexpr (END == END_STORE && sizeof(T) == 2) {
        if (c.M <= 32) return launch_ring_x<4, TOut, SW, END, T>(c, p, stream);
        return launch_ring_x<8, TOut, SW, END, T>(c, p, stream);
    }
    TL_REQUIRE(false, "gemm_ring: too many rows (%d)", c.M);
}

// Which kernel a bfloat16 product of aligned operands and up to 64 rows gets, K a multiple of 64 (for tests): 0 the rings, 1 the few-rows kernel that fetches into registers, 2 tiles.
// `gated`: N outputs of the fused gate.
extern "C" int tl_gemm_few_rows_choice(int M, int N, int K, int gated) {
    if (gated) return ring_pays_gated(M, N, K) ? 0 : M <= 16 ? 1 : 2;
    return ring_pays(M, N, K) ? 0 : M > 8 ? 2 : 1;
}

// The plan of a product through the rings (for tests): `halves` 2 for the fused gate; K in `parts` ranges.
extern "C" void tl_gemm_ring_plan(int total, int M, int K, int halves, int units, int even, int parts, int* wj, int* rows) {
    const RingPlan p = plan_ring(total, M, halves, units / parts, even != 0, ring_spread(K), parts > 1);
    *wj = p.wj;
    *rows = p.rows;
}

// The same in 32 bits; `pairs`: rows by pairs, `total` of them.
extern "C" void tl_gemm_f32_ring_plan(int total, int M, int K, int pairs, int units, int* wj, int* rows) {
    const RingPlan p = plan_ring(total, M, pairs ? 2 : 1, units, false, ring_spread<float>(K), false, pairs != 0);
    *wj = p.wj;
    *rows = p.rows;
}

// One shape of the kernel above (for tests and tuning): 8 wj weight rows a work-group (with `gate`, 1 + the gate's number, half gate and half up rows), `rows` outputs of which
// are used; parts > 1: K split into ranges of k_per columns, float slabs.  wj 0: as the dispatch would.
extern "C" int tl_gemm_ring_variant(const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int N, int K, int ldx, int ldo, int out_f32, int gate, int wj,
                                    int rows, int parts, int k_per, hipStream_t stream) {
    const int total = gate ? ldo : N, halves = gate ? 2 : 1;
    TL_REQUIRE(ring_fits(x, w, M, K, ldx) && N > 0 && ldo >= (gate ? 1 : N) && gate >= 0 && gate <= 3 && (!gate || (!out_f32 && N == (ldo + 31) / 32 * 64)),
               "gemm_ring: bad sizes M=%d N=%d K=%d", M, N, K);
    TL_REQUIRE(wj == 0 || (wj > 0 && wj <= 8 && rows > 0 && rows <= 8 * wj / halves), "gemm_ring: %d outputs do not fit %d requests", rows, wj);
    TL_REQUIRE(parts == 1 || (parts > 1 && out_f32 && !bias && k_per > 0 && k_per % 64 == 0 && (long)k_per * (parts - 1) < K && (long)k_per * parts >= K),
               "gemm_ring: %d ranges of %d columns are not a split of %d", parts, k_per, K);
    RingCall c{x, w, bias, bias_f32, out, M, N, K, ldx, ldo, gate ? total : 0, parts, parts > 1 ? k_per : 0};
    const RingPlan p{wj, rows};
    if (gate == 1) return launch_ring<bf16_t, 1, END_STORE>(c, stream, p);
    if (gate == 2) return launch_ring<bf16_t, 2, END_STORE>(c, stream, p);
    if (gate == 3) return launch_ring<bf16_t, 3, END_STORE>(c, stream, p);
    return out_f32 ? launch_ring<float, 0, END_STORE>(c, stream, p) : launch_ring<bf16_t, 0, END_STORE>(c, stream, p);
}

// One named kernel of the 32-bit products (for tests and tuning), or an error where it is not built for the sizes: 0 the general tile kernel (v_fma_f32), 1 the matrix-core
// tile kernel, 2 and 3 the kernels for few rows on multiply-adds (up to 8) and on the matrix cores (up to 16), 4 to 6 the matrix-core tile kernel with tiles of 64 x 64, 64 x 128, 128 x 128,
// 7 and 8 with 64 x 32 and 32 x 32, 9 the rings (wj > 0: in shapes of wj requests, `rows` outputs of them used).
extern "C" int tl_gemm_f32_variant(const void* x, const void* w, const void* bias, int bias_f32, void* out,
                                   int M, int N, int K, int ldx, int ldo, int matrix_cores, int wj, int rows, hipStream_t stream) {
    TL_REQUIRE(M > 0 && N > 0 && K > 0 && ldx >= K && ldo >= N, "gemm_f32: bad sizes M=%d N=%d K=%d ldx=%d ldo=%d", M, N, K, ldx, ldo);
    TL_REQUIRE(matrix_cores >= 0 && matrix_cores <= 9, "gemm_f32: no kernel %d", matrix_cores);
    if (matrix_cores == 9) {
        TL_REQUIRE(ring_fits_f32(x, w, M, K, ldx), "gemm_f32: the rings need M <= 16, K %% 32 == 0 and 16-byte aligned rows");
        TL_REQUIRE(wj <= 0 || (wj <= 8 && rows > 0 && rows <= 8 * wj), "gemm_f32: %d outputs do not fit %d requests", rows, wj);
        return launch_ring<float, 0, END_STORE, float>(RingCall{x, w, bias, bias_f32, out, M, N, K, ldx, ldo, 0}, stream, RingPlan{max(wj, 0), rows});
    }
    if (matrix_cores == 2 || matrix_cores == 3) {
        TL_REQUIRE(gemv_f32_fits(x, w, M, K, ldx) && (matrix_cores == 3 || M <= 8), "gemm_f32: the few-rows kernels need M <= 8 or 16, K %% 4 == 0 and 16-byte aligned rows");
        if (matrix_cores == 2) launch_gemv_f32_fma<F32_PLAIN>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, F32Pairs{}, stream);
        else launch_gemv_f32_mfma(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, stream);
    } else if (matrix_cores) {
        TL_REQUIRE(gemm_f32_mfma_fits(x, w, 17, K, ldx), "gemm_f32: the matrix-core kernel needs K %% 4 == 0 and 16-byte aligned rows");
        launch_gemm_f32_mfma(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, stream, matrix_cores > 3 ? matrix_cores - 3 : 0);
    } else {
        launch_gemm_tile<float, float>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, stream);
    }
    TL_CHECK_LAUNCH("gemm_f32");
    return TL_OK;
}

// One named instance of the few-rows kernel, of those the dispatch below can pick (for tests and tuning);
// rows_per_strip: 0 for strips of 16 R rows, else that many (at most 16 R).
extern "C" int tl_gemm_skinny_variant(const void* x, const void* w, const void* bias, int bias_f32, void* out,
                                      int M, int N, int K, int ldx, int ldo, int out_f32, int R, int KS, int rows_per_strip,
                                      hipStream_t stream) {
    TL_REQUIRE(M > 0 && M <= 64 && K % 8 == 0 && ldx % 8 == 0, "gemm_skinny: needs 0 < M <= 64 and K, ldx multiples of 8");
    TL_REQUIRE(rows_per_strip >= 0 && rows_per_strip <= 16 * R, "gemm_skinny: a strip of %d blocks holds up to %d rows, not %d", R, 16 * R, rows_per_strip);
    const int MT = M <= 16 ? 1 : (M <= 32 ? 2 : 4);
#define TL_SKINNY_CASE(r, t, k) \
    if (R == r && MT == t && KS == k) { launch_skinny<r, t, k>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_f32, stream, rows_per_strip); TL_CHECK_LAUNCH("gemm_skinny"); return TL_OK; }
    // the instances pick_skinny can choose
    TL_SKINNY_CASE(1, 1, 16) TL_SKINNY_CASE(1, 2, 16) TL_SKINNY_CASE(1, 1, 8) TL_SKINNY_CASE(1, 2, 8) TL_SKINNY_CASE(2, 1, 8)
    TL_SKINNY_CASE(4, 4, 4) TL_SKINNY_CASE(2, 4, 2) TL_SKINNY_CASE(1, 4, 8)
#undef TL_SKINNY_CASE
    TL_REQUIRE(false, "gemm_skinny: no instance R=%d MT=%d KS=%d", R, MT, KS);
}

// =====================================================================================
// bfloat16 on the matrix cores, many rows (prompt portions): shared-memory tiles.
//
// A work-group of four or eight waves owns a BM x BN tile of the output and walks K in slabs of TK
// (32 or 64) elements.
// A slab of x (BM rows) and of w (BN rows) is fetched from memory as 16-byte pieces into
// registers while the previous slab is being multiplied, then parked in shared memory
// (two buffers, one barrier per slab).  Rows lie 2 TK + 16 bytes apart in shared memory (16 of
// padding) so that the 16-byte operand reads of v_mfma_f32_32x32x16_bf16 do not
// collide on banks.  Waves are laid out WGM x WGN over the tile; each multiplies
// (BM / WGM) x (BN / WGN) as blocks of 32 x 32 with float accumulators.
// Needs K % 8 == 0 and 16-byte aligned rows.

// Which tile a shape gets (measured on MI355X at Qwen2.5-7B sizes, 2048 and 512 rows):
//   * 256 x 256 with slabs of 64 (eight waves) reuses operands best (840 TFLOP/s on the
//     gate/up product) but needs over a thousand such tiles to keep 256 compute units busy;
//   * otherwise 128 x 128 with slabs of 64 (two work-groups fit a compute unit: 512 at once),
//     except when the tile count lies between 512 and 768, where slabs of 32 (three fit) avoid
//     a second, nearly empty round;
//   * up to 64 rows: 64 x 128.
enum TileChoice { TILE_64x128, TILE_128x128_K32, TILE_128x128_K64, TILE_256x256 };
static TileChoice pick_tile(int M, int N) {
    if (M <= 64) return TILE_64x128;
    const long big = (long)((M + 255) / 256) * ((N + 255) / 256);
    if (big >= 1024) return TILE_256x256;
    const long wgs = (long)((M + 127) / 128) * ((N + 127) / 128);
    if (wgs > 512 && wgs <= 768) return TILE_128x128_K32;
    return TILE_128x128_K64;
}

template <int BM, int BN, int WGM, int WGN, typename TOut, int SW = 0, int TK = 32>
__global__ __launch_bounds__(64 * WGM * WGN) void gemm_mfma_tile_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                             const void* __restrict__ bias, int bias_f32,
                                                             TOut* __restrict__ out, int M, int N, int K, int ldx, int ldo,
                                                             int out_cols = 0) {
    static_assert(!SW || (BN / WGN) % 64 == 0, "the fused gate needs whole 64-row blocks per wave");
    constexpr int TROW = TK + 8;                         // elements between rows in shared memory (16 bytes of padding)
    constexpr int NT = 64 * WGM * WGN;                   // threads
    constexpr int WM = BM / WGM, WN = BN / WGN;          // wave tile
    constexpr int FM = WM / 32, FN = WN / 32;            // 32x32 blocks per wave
    constexpr int PIECES = (BM + BN) * (TK / 8);         // 16-byte pieces per slab
    constexpr int PPT = PIECES / NT;                     // pieces per thread
    static_assert(PIECES % NT == 0, "slab must divide over the threads");
    extern __shared__ __attribute__((aligned(16))) bf16_t lds_raw[];
    bf16_t (*lds)[(BM + BN) * TROW] = (bf16_t (*)[(BM + BN) * TROW])lds_raw;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WGN, wn = wave % WGN;
    // Which tile this work-group owns.  Work-groups are dealt to the 8 XCDs round-robin by
    // blockIdx, and each XCD has an L2 of its own: give every XCD a contiguous range of
    // "logical" tile numbers, and number tiles so that 64 consecutive ones (what an XCD runs at
    // a time) form an 8 x 8 block of the output, so that each operand tile it fetches is used
    // by eight work-groups out of its L2.
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    int lid;
    {
        const int total = gridDim.x, xcd = blockIdx.x % 8, idx = blockIdx.x / 8;
        lid = xcd * (total / 8) + min(xcd, total % 8) + idx;
    }
    int tm, tn;
    {
        const int per_group = 8 * tiles_n;
        const int first_m = (lid / per_group) * 8;
        const int rows = min(tiles_m - first_m, 8);
        tm = first_m + (lid % per_group) % rows;
        tn = (lid % per_group) / rows;
    }
    const int m0 = tm * BM, n0 = tn * BN;

    // which pieces this thread fetches: piece p -> (row, 8-element column) of the stacked [x rows; w rows] slab
    const bf16_t* src[PPT];
    int dst[PPT];
    int kcol[PPT];
#pragma unroll
    for (int i = 0; i < PPT; ++i) {
        const int p = tid + i * NT;
        const int row = p / (TK / 8), c = p % (TK / 8);
        kcol[i] = c * 8;
        dst[i] = row * TROW + c * 8;
        if (row < BM) src[i] = x + (size_t)min(m0 + row, M - 1) * ldx + c * 8;
        else src[i] = w + (size_t)min(n0 + row - BM, N - 1) * K + c * 8;
    }

    f32x16_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    const int slabs = (K + TK - 1) / TK;
    uint4 stage[PPT];
#pragma unroll
    for (int i = 0; i < PPT; ++i) stage[i] = (kcol[i] + 8 <= K) ? *(const uint4*)(src[i]) : make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < PPT; ++i) *(uint4*)(&lds[0][dst[i]]) = stage[i];
    __syncthreads();

    const int fr = lane & 31, fk = (lane >> 5) * 8;      // operand fragment: row within block, k offset
    for (int sl = 0; sl < slabs; ++sl) {
        const int cur = sl & 1;
        if (sl + 1 < slabs) {
            const int k0 = (sl + 1) * TK;
#pragma unroll
            for (int i = 0; i < PPT; ++i)
                stage[i] = (k0 + kcol[i] + 8 <= K) ? *(const uint4*)(src[i] + k0) : make_uint4(0, 0, 0, 0);
        }
        const bf16_t* xs = &lds[cur][0];
        const bf16_t* ws = &lds[cur][BM * TROW];
#pragma unroll
        for (int kk = 0; kk < TK; kk += 16) {
            Frag16 af[FM], bfr[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i) af[i].u = *(const uint4*)(xs + (wm * WM + i * 32 + fr) * TROW + kk + fk);
#pragma unroll
            for (int j = 0; j < FN; ++j) bfr[j].u = *(const uint4*)(ws + (wn * WN + j * 32 + fr) * TROW + kk + fk);
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i].v, bfr[j].v, acc[i][j], 0, 0, 0);
        }
        if (sl + 1 < slabs) {
#pragma unroll
            for (int i = 0; i < PPT; ++i) *(uint4*)(&lds[cur ^ 1][dst[i]]) = stage[i];
        }
        __syncthreads();
    }

    // block result: lane holds column (lane % 32), rows 8 * (v / 4) + 4 * (lane / 32) + v % 4
    if (SW) {   // even blocks hold gate columns, the next block the up columns of the same outputs
#pragma unroll
        for (int j = 0; j + 1 < FN; j += 2) {
            const int col = (n0 + wn * WN + j * 32) / 2 + (lane & 31);
            if (col >= out_cols) continue;
#pragma unroll
            for (int i = 0; i < FM; ++i) {
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int m = m0 + wm * WM + i * 32 + 8 * (v / 4) + 4 * (lane >> 5) + (v % 4);
                    if (m < M) out[(size_t)m * ldo + col] = from_float<TOut>(gate_mul<SW>(acc[i][j][v], acc[i][j + 1][v]));
                }
            }
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int n = n0 + wn * WN + j * 32 + (lane & 31);
        if (n >= N) continue;
        const float b = bias ? load_vec(bias, bias_f32, n) : 0.f;
#pragma unroll
        for (int i = 0; i < FM; ++i) {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int m = m0 + wm * WM + i * 32 + 8 * (v / 4) + 4 * (lane >> 5) + (v % 4);
                if (m < M) out[(size_t)m * ldo + n] = from_float<TOut>(acc[i][j][v] + b);
            }
        }
    }
}

// Shared memory of a tile kernel: two buffers of (BM + BN) rows of TK + 8 elements.

template <int BM, int BN, int WGM, int WGN, typename TOut, int SW, int TK>
static int launch_mfma_tile_t(const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int N, int K,
                              int ldx, int ldo, int out_cols, hipStream_t stream) {
    constexpr size_t lds = 2 * (size_t)(BM + BN) * (TK + 8) * sizeof(bf16_t);
    auto kernel = gemm_mfma_tile_kernel<BM, BN, WGM, WGN, TOut, SW, TK>;
    static hipError_t allowed = allow_lds(kernel, lds);
    if (allowed != hipSuccess) {
        tl_set_error("gemm_mfma_tile: cannot get %zu bytes of shared memory: %s", lds, hipGetErrorString(allowed));
        return TL_ERR_HIP;
    }
    dim3 grid(((M + BM - 1) / BM) * ((N + BN - 1) / BN)), block(64 * WGM * WGN);
    kernel<<<grid, block, lds, stream>>>((const bf16_t*)x, (const bf16_t*)w, bias, bias_f32, (TOut*)out, M, N, K, ldx, ldo, out_cols);
    return TL_OK;
}

template <int BM, int BN, int WGM, int WGN, int TK = 32>
static int launch_mfma_tile(const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int N, int K,
                            int ldx, int ldo, int out_f32, hipStream_t stream) {
    if (out_f32) return launch_mfma_tile_t<BM, BN, WGM, WGN, float, false, TK>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, 0, stream);
    return launch_mfma_tile_t<BM, BN, WGM, WGN, bf16_t, false, TK>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, 0, stream);
}

// Tile shapes of the direct-load kernel and which one a product gets.  Estimate per shape: the
// tiles are dealt to 256 compute units, each works through ceil(tiles / 256) of them one after
// the other; a tile takes a fixed time (filling the pipeline, storing the result) plus its
// products at the rate one compute unit reaches with that shape.  The figures are fitted to measurements of every shape at 16 to 8192 rows
// against 27 matrices (the Qwen2.5 models' and those 2048 to 16384 wide of the other designs; the rates of 64 x 192, 64 x 320 and 256 x 320 came out as they were): a whole
// product gets a shape whose time is 1.005 of the fastest shape's on average over those 341 sizes, 1.13 at most, and 1.008 over 160 others, 1.14 at most
// (1.07 and 1.8 with the figures fitted to 2048 rows alone).
// (DL_128x128_S4: 128 x 128 with four slabs in shared memory, one work-group to a compute unit: where the tiles are one round of work-groups, what
// counts is how many bytes a work-group has on their way: 2048 x 2048 x 8192 69.6 us against 102.7 with two slabs, 2048 x 2048 x 2048 21.1 against 25.9, 400 x 7168 x 5120
// 1.8 times as fast; with more tiles than units two work-groups of two slabs each share a unit: 2048 x 8192 x 2048 65.5 us against 75.2)
// (DL_256x320: eight waves of 64 x 160, 250 registers, 144 KB of slabs; float slabs of a split K only, since a bfloat16
// result tile of 160 KB does not fit its slab buffers.  It is there for thousands of rows against a matrix 5120 wide:
// 2048 rows are 160 tiles of 256 x 256, which leave 96 of 256 compute units idle, and 128 of these, which with K in
// two halves are one round of 256 work-groups.  Measured at 2048 rows, slabs written: 5120 x 27648 430 us against
// 480 in three parts of 256 x 256 and 546 in two of 256 x 160; 5120 x 13824 218 against 259 and 280.)
// (DL_256x160: four waves of 64 x 160, for matrices 5120 wide as well: 2048 rows are 256 tiles, one to a compute
// unit, and 4096 rows two rounds of them where tiles of 256 x 256 take one and a quarter.  A compute unit gets through
// a slab of it hardly faster than through one of 256 x 256 (what a slab costs is mostly its requests, 52 against 64,
// not its products, 40 against 64), so it wins only where it fills rounds that the square tile leaves part empty.)
// (Tiles of 256 x 224, which fill the rounds of matrices 3584 and 7168 wide, are at most 4 % faster than the best of these anywhere: a chip with
// idle compute units runs the others at a higher clock.)
enum DlTile { DL_64x64, DL_64x256, DL_128x128, DL_128x256, DL_256x128, DL_192x256, DL_256x192, DL_256x256, DL_64x128, DL_128x128_S4, DL_64x192, DL_128x192, DL_64x320, DL_256x320, DL_256x160, DL_TILES };
static const int DL_BM[DL_TILES] = {64, 64, 128, 128, 256, 192, 256, 256, 64, 128, 64, 128, 64, 256, 256};
static const int DL_BN[DL_TILES] = {64, 256, 128, 256, 128, 256, 192, 256, 128, 128, 192, 192, 320, 320, 160};

// Seconds for `groups` work-groups of tile t over k columns each.  The two smallest tiles run two
// to a compute unit: each then works at half the unit's rate, and one that has a unit to itself
// (not more work-groups than units) at about 0.87 of it.  With few rows the products wait for the
// operands: a compute unit fills its shared memory at about 69 GB/s, and a work-group draws its BN
// rows of weights and its BM rows of x alike (x as often as there are tiles along N: with 64 x 64 tiles
// as many bytes of x as of weights).  Measured at 64 rows: on the 14B's gate/up matrix 108 work-groups
// of 64 x 256 take 80 us, 216 of 64 x 128 59, 432 of 64 x 64 (two to a unit) 68.
struct DlFigures {
    double rate[DL_TILES], fixed[DL_TILES];      // FLOP/s of one compute unit; seconds per tile
    double stream, alone, lag;                   // bytes per second of a compute unit; see above; a factor on single rounds of 128 x 128
    bool x_counts;                               // whether the rows of x count as bytes that a work-group draws
};
static double dl_estimate(const DlFigures& f, DlTile t, long groups, int k) {
    const bool pairs = t == DL_64x64 || t == DL_128x128;
    const double products = 2.0 * DL_BM[t] * DL_BN[t] * k;
    const double stream = 2.0 * (DL_BN[t] + (f.x_counts ? DL_BM[t] : 0)) * k / f.stream;
    const int cus = TL_COMPUTE_UNITS;
    if (!pairs) return (double)((groups + cus - 1) / cus) * fmax(products / f.rate[t] + f.fixed[t], stream);
    const double rate = f.rate[t] * (groups > cus ? 0.5 : f.alone);
    const double lag = t == DL_128x128 && groups <= 2 * cus ? f.lag : 1.0;
    return lag * (double)((groups + 2 * cus - 1) / (2 * cus)) * fmax(products / rate + f.fixed[t], groups > cus ? 2 * stream : stream);
}
static const DlFigures DL_NOW = {
    {2.52e12, 2.82e12, 3.71e12, 4.41e12, 5.38e12, 4.34e12, 5.27e12, 6.23e12, 1.89e12, 4.01e12, 3.0e12, 4.83e12, 3.5e12, 5.5e12, 4.48e12},
    {2.7e-6, 9.5e-6, 5.5e-6, 11e-6, 8.4e-6, 11e-6, 9.1e-6, 15.4e-6, 3.1e-6, 5.2e-6, 9.7e-6, 10.6e-6, 12e-6, 5.1e-6, 10.6e-6}, 68.8e9, 0.87, 1.0, true};
// The numbers of the rule by which a product's result stays in 32 bits (gives_slabs below).  They are no kernel's: they were the estimates of slower kernels when the line was drawn, and stay, since
// a result that a consumer has read in 32 bits is not to lose them because a tile has become faster.
static const DlFigures DL_SLAB_RULE = {
    {2.45e12, 3.3e12, 4.2e12, 4.6e12, 4.8e12, 5.2e12, 5.2e12, 6.1e12, 2.1e12, 4.2e12, 3.0e12, 4.4e12, 3.5e12, 5.5e12, 4.3e12},
    {2.7e-6, 11.5e-6, 5.5e-6, 11e-6, 15e-6, 6e-6, 8e-6, 14e-6, 5e-6, 4.5e-6, 9e-6, 9e-6, 12e-6, 10e-6, 10e-6}, 32e9, 0.62, 1.1, false};

static long dl_tiles(DlTile t, int M, int N) { return (long)((M + DL_BM[t] - 1) / DL_BM[t]) * ((N + DL_BN[t] - 1) / DL_BN[t]); }

static DlTile pick_dl_tile(int M, int N, int K, bool sw, int products = 1) {
    DlTile best = DL_128x128;
    double best_t = 1e30;
    for (int t = 0; t < DL_TILES; ++t) {
        if (sw && (t == DL_64x64 || t == DL_256x192 || t == DL_64x320 || t == DL_256x160)) continue;      // a wave of the fused gate needs whole 64-row blocks of weights
        if (t == DL_256x320) continue;      // float slabs of partial sums only: a bfloat16 result tile of 160 KB does not fit its slab buffers
        const long tiles = dl_tiles((DlTile)t, M, N) * products;
        if (t == DL_128x128_S4 && tiles > TL_COMPUTE_UNITS) continue;      // one round of work-groups
        double est = dl_estimate(DL_NOW, (DlTile)t, tiles, K);
        // One row of tiles: no weight is drawn twice, all come from memory and none from the L2s, and there the small tile with two work-groups on some of the units, and the deep one with
        // the fused gate, fall behind their estimates.  Measured (us; 64 x 64 / 64 x 128 / 128 x 128 with four slabs): 63 x 18944 x 5120 62.5 / 52.9 / 52.5, 63 x 18944 x 3584 40.7 / 37.1 /
        // 36.3, 33 x 22528 x 5120 57.4 / 51.4 / 50.6; where rows of w lie multiples of 4 KB apart, or are short, the small tile stays ahead (33 x 27648 x 8192 91 / 105 / 102, x 768 12.4 / 13.0 / 13.0); the gate, 128 x
        // 5632 x 13824 - / 113 / 137, 128 x 6912 x 5120 - / 48.7 / 58.0.  (Without these two lines 94 of 1134 sizes of 33 to 700 rows took more than 3 % longer, up to 19 %, than
        // with the shapes that the rule before the figures above chose, with them 55, up to 14 %; of 427 with the gate 15, up to 21 %, and 6, up to 13 %.)
        if (t == DL_64x64 && M <= 64 && tiles > TL_COMPUTE_UNITS && K > 2048 && K % 2048) est *= 1.4;
        if (t == DL_128x128_S4 && sw && M > 64 && M <= 128) est *= 1.05;
        if (est < best_t) { best_t = est; best = (DlTile)t; }
    }
    return best;
}

// The tile of a whole product (gated: with the fused gate, N rows of its interleaved matrix), by its rows, columns and slabs in shared memory; tests ask for it.
extern "C" void tl_gemm_direct_choice(int M, int N, int K, int gated, int* rows, int* columns, int* slabs4) {
    const DlTile t = pick_dl_tile(M, N, K, gated != 0);
    *rows = DL_BM[t];
    *columns = DL_BN[t];
    *slabs4 = t == DL_128x128_S4;
}

// K in `parts` ranges of k_per columns (a multiple of 64), none of them empty; 0 if there is no such split.
static int dl_k_per(int K, int parts) {
    const int k_per = ((K / 64 + parts - 1) / parts) * 64;
    return (K + k_per - 1) / k_per == parts ? k_per : 0;
}
static const DlTile DL_ALONE[] = {DL_128x128_S4, DL_128x256, DL_256x128, DL_192x256, DL_256x192, DL_256x256, DL_256x320, DL_64x64};      // a compute unit to themselves
static bool dl_can_split(DlTile t, int M, int N, int parts, int small_rows) {
    const bool one_round = dl_tiles(t, M, N) * parts <= TL_COMPUTE_UNITS;
    // (the small tile as for up to 64 rows, one work-group to a compute unit: 128 rows against the 7B's output
    // projection 13.0 us in two parts where four parts of 128 x 128 take 17.0)
    return t == DL_128x128_S4 ? one_round : t == DL_64x64 ? one_round && M <= small_rows : true;
}

// Whether a product of more than 64 rows whose consumer can add slabs up gives it float slabs: a line between the sizes whose sums reach the consumer in 32 bits and those that are rounded
// to bfloat16 first, drawn where K split over work-groups was ahead of a bfloat16 result.  What it costs by today's times, product and reading against the best whole product with a bfloat16 result:
// 512 rows against 5120 x 13824 0.67, 5120 x 5120 0.84, 7168 x 5120 0.99; over 574 sizes on its yes side 0.84 on average; 75 of them are more than 5 % behind, up to 1.35 (1457 x 2048 x 4096),
// mostly where the plan below splits what one slab would do faster.
static bool gives_slabs(int M, int N, int K) {
    double whole = 1e30;
    for (int t = 0; t < DL_TILES; ++t) {
        if (t == DL_256x320 || t == DL_64x192 || t == DL_128x192 || t == DL_64x320) continue;
        const long tiles = dl_tiles((DlTile)t, M, N);
        if (t == DL_128x128_S4 && (tiles > TL_COMPUTE_UNITS || M > 128)) continue;
        whole = fmin(whole, dl_estimate(DL_SLAB_RULE, (DlTile)t, tiles, K));
    }
    whole += (double)M * N * 2 * 2 / 3e12;
    for (DlTile t : DL_ALONE)
        for (int P = 2; P <= 8 && K / P >= 512; ++P) {
            const int k_per = dl_k_per(K, P);
            if (k_per && dl_can_split(t, M, N, P, 128) &&
                1.1 * dl_estimate(DL_SLAB_RULE, t, dl_tiles(t, M, N) * P, k_per) + (double)P * M * N * 4 * 2 / 3e12 < whole) return true;
        }
    return false;
}

// More than 64 rows against a matrix whose output tiles leave compute units idle (a few hundred rows
// of a prompt portion against the down projection, say): K split over `parts` work-groups per tile
// into float slabs that the consumer adds up, or one float slab where a tile's own rounds fill the chip better (400 x 7168 x 3584: 34.2 us in two parts of 256 x 128, 29.7 in one of
// 128 x 128 with four slabs in shared memory; 133 x 4608 x 3584 16.5 in three parts, 14.6 in one of 64 x 64).  Split, only the tiles that have a compute unit to themselves
// are considered; the slabs cost their bytes once written and once read.  parts == 0: a bfloat16 result.
// With the slabs' reading counted at 4 TB/s the choice takes 1.026 of the fastest plan's time on average over 123 of the fitted sizes, 1.28 at most, and 1.078 over 51 others, 1.54 at most:
// it undervalues one slab of 128 x 128 (1457 x 2048 x 4096 34.6 in two parts, 28.6 in one).  Against the plans before the tiles' figures were refitted, the norm that adds the slabs up included: 0.97 on average over
// 410 sizes of 65 to 700 rows, 33 of them more than 3 % slower, up to 1.16 (133 x 4608 x 8192: seven parts of 256 x 128 where three of 128 x 128 would take 0.82 of that); no factor on one shape or on one
// slab that mends those leaves the others as they are.
struct DlSplit { DlTile tile; int parts; int k_per; };
static DlSplit plan_dl_split(int M, int N, int K) {
    DlSplit best{DL_128x128, 0, 0};
    if (!gives_slabs(M, N, K)) return best;
    double best_t = 1e30;
    auto consider = [&](DlTile t, int P, int k_per) {
        // (a tenth on top: float slabs leave the kernel more slowly than the estimate's bfloat16 rows)
        const double est = 1.11 * dl_estimate(DL_NOW, t, dl_tiles(t, M, N) * P, k_per) + (double)P * M * N * 5.9 / 3e12;
        if (est < best_t) { best_t = est; best = DlSplit{t, P, k_per}; }
    };
    for (int t = 0; t < DL_TILES; ++t)
        if (t != DL_128x128_S4 || dl_tiles((DlTile)t, M, N) <= TL_COMPUTE_UNITS) consider((DlTile)t, 1, K);
    for (DlTile t : DL_ALONE)
        for (int P = 2; P <= 8 && K / P >= 512; ++P) {
            const int k_per = dl_k_per(K, P);
            if (k_per && dl_can_split(t, M, N, P, 256)) consider(t, P, k_per);
        }
    return best;
}

// parts > 1 (float results only): K is split into `parts` ranges of k_per columns and out holds that many [M, ldo] slabs.
template <int BM, int BN, int WGM, int WGN, int STAGES, typename TOut, int SW>
static int launch_dl_tile_t(const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int N, int K,
                            int ldx, int ldo, int out_cols, hipStream_t stream, int parts = 1, int k_per = 0, Groups gr = Groups{}) {
    constexpr size_t lds = (size_t)STAGES * dl_slab_rows(BM, BN, WGM * WGN) * 64 * sizeof(bf16_t);
    // (a lane's offset from its tile's first row is kept in 32 bits)
    TL_REQUIRE((long)(BM > BN ? BM : BN) * (ldx > K ? ldx : K) * 2 < (1L << 31), "gemm_dl_tile: rows of %d elements are too long", ldx > K ? ldx : K);
    auto kernel = gemm_dl_tile_kernel<BM, BN, WGM, WGN, STAGES, TOut, SW>;
    static hipError_t allowed = allow_lds(kernel, lds);
    if (allowed != hipSuccess) {
        tl_set_error("gemm_dl_tile: cannot get %zu bytes of shared memory: %s", lds, hipGetErrorString(allowed));
        return TL_ERR_HIP;
    }
    dim3 grid(((M + BM - 1) / BM) * ((N + BN - 1) / BN), parts, gr.count), block(64 * WGM * WGN);
    kernel<<<grid, block, lds, stream>>>((const bf16_t*)x, (const bf16_t*)w, bias, bias_f32, (TOut*)out, M, N, K, ldx, ldo, out_cols,
                                         parts > 1 ? k_per : 0, gr.stride);
    return TL_OK;
}

template <typename TOut, int SW>
static int launch_dl_tile(DlTile tile, const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int N, int K,
                          int ldx, int ldo, int out_cols, hipStream_t stream, int parts = 1, int k_per = 0, Groups gr = Groups{}) {
    switch (tile) {
    case DL_64x64:
        if constexpr (!SW) return launch_dl_tile_t<64, 64, 2, 2, 4, TOut, false>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_cols, stream, parts, k_per, gr);
        else break;
    case DL_64x256: return launch_dl_tile_t<64, 256, 1, 4, 3, TOut, SW>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_cols, stream, parts, k_per, gr);
    case DL_128x128: return launch_dl_tile_t<128, 128, 2, 2, 2, TOut, SW>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_cols, stream, parts, k_per, gr);
    case DL_128x128_S4: return launch_dl_tile_t<128, 128, 2, 2, 4, TOut, SW>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_cols, stream, parts, k_per, gr);
    case DL_128x256: return launch_dl_tile_t<128, 256, 2, 4, 3, TOut, SW>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_cols, stream, parts, k_per, gr);
    case DL_256x128: return launch_dl_tile_t<256, 128, 4, 2, 3, TOut, SW>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_cols, stream, parts, k_per, gr);
    case DL_64x128: return launch_dl_tile_t<64, 128, 1, 2, 3, TOut, SW>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_cols, stream, parts, k_per, gr);
    case DL_64x192: return launch_dl_tile_t<64, 192, 1, 3, 4, TOut, SW>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_cols, stream, parts, k_per, gr);
    case DL_64x320:
        if constexpr (!SW) return launch_dl_tile_t<64, 320, 1, 5, 3, TOut, false>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_cols, stream, parts, k_per, gr);
        else break;
    case DL_128x192: return launch_dl_tile_t<128, 192, 2, 3, 3, TOut, SW>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_cols, stream, parts, k_per, gr);
    case DL_192x256: return launch_dl_tile_t<192, 256, 2, 4, 2, TOut, SW>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_cols, stream, parts, k_per, gr);
    case DL_256x192:
        if constexpr (!SW) return launch_dl_tile_t<256, 192, 4, 2, 2, TOut, false>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_cols, stream, parts, k_per, gr);
        else break;
    case DL_256x256: return launch_dl_tile_t<256, 256, 2, 4, 2, TOut, SW>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_cols, stream, parts, k_per, gr);
    case DL_256x160:
        if constexpr (!SW) return launch_dl_tile_t<256, 160, 4, 1, 2, TOut, false>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_cols, stream, parts, k_per, gr);
        else break;
    case DL_256x320:
        if constexpr (!SW && sizeof(TOut) == 4) return launch_dl_tile_t<256, 320, 4, 2, 2, float, false>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_cols, stream, parts, k_per, gr);
        else break;
    default: break;
    }
    tl_set_error("gemm_dl_tile: no instance of tile %d", (int)tile);
    return TL_ERR_ARG;
}

// One named tile shape of the many-rows kernel (tests cover each; tuning times them).
extern "C" int tl_gemm_tile_variant(const void* x, const void* w, const void* bias, int bias_f32, void* out,
                                    int M, int N, int K, int ldx, int ldo, int out_f32, int BM, int BN, int TK, hipStream_t stream) {
    TL_REQUIRE(M > 0 && K % 8 == 0 && ldx % 8 == 0, "gemm_tile: needs M > 0 and K, ldx multiples of 8");
    int rc = -1;
#define TL_TILE_CASE(bm, bn, gm, gn, tk) \
    if (BM == bm && BN == bn && TK == tk) rc = launch_mfma_tile<bm, bn, gm, gn, tk>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_f32, stream);
    // the tile shapes pick_tile can choose
    TL_TILE_CASE(128, 128, 2, 2, 32) TL_TILE_CASE(128, 128, 2, 2, 64)
    TL_TILE_CASE(64, 128, 2, 2, 64) TL_TILE_CASE(256, 256, 4, 2, 64)
#undef TL_TILE_CASE
    TL_REQUIRE(rc != -1, "gemm_tile: no instance BM=%d BN=%d TK=%d", BM, BN, TK);
    if (rc != TL_OK) return rc;
    TL_CHECK_LAUNCH("gemm_mfma_tile");
    return TL_OK;
}

// One named tile shape of the direct-load kernel (tests cover each; tuning times them).
extern "C" int tl_gemm_direct_variant(const void* x, const void* w, const void* bias, int bias_f32, void* out,
                                      int M, int N, int K, int ldx, int ldo, int out_f32, int BM, int BN, hipStream_t stream) {
    TL_REQUIRE(M > 0 && K % 64 == 0 && ldx % 8 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0,
               "gemm_direct: needs M > 0, K a multiple of 64 and 16-byte aligned rows");
    int tile = -1;
    for (int t = 0; t < DL_TILES; ++t)
        if (DL_BM[t] == BM && DL_BN[t] == BN && t != DL_128x128_S4) tile = t;
    TL_REQUIRE(tile >= 0, "gemm_direct: no tile of %d x %d", BM, BN);
    const int rc = out_f32 ? launch_dl_tile<float, false>((DlTile)tile, x, w, bias, bias_f32, out, M, N, K, ldx, ldo, 0, stream)
                           : launch_dl_tile<bf16_t, false>((DlTile)tile, x, w, bias, bias_f32, out, M, N, K, ldx, ldo, 0, stream);
    if (rc != TL_OK) return rc;
    TL_CHECK_LAUNCH("gemm_dl_tile");
    return TL_OK;
}

// The fused gate/up product (see tl_gemm_swiglu) on one named tile shape; for tests and tuning.
extern "C" int tl_gemm_swiglu_direct_variant(const void* x, const void* w, void* out, int M, int I, int K, int ldx, int ldo,
                                             int BM, int BN, hipStream_t stream) {
    TL_REQUIRE(M > 0 && I > 0 && K % 64 == 0 && ldx % 8 == 0 && ldo >= I && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0,
               "gemm_swiglu_direct: needs M > 0, K a multiple of 64 and 16-byte aligned rows");
    int tile = -1;
    for (int t = 0; t < DL_TILES; ++t)
        if (DL_BM[t] == BM && DL_BN[t] == BN && t != DL_128x128_S4 && t != DL_64x64 && t != DL_256x192 && t != DL_64x320 && t != DL_256x320 && t != DL_256x160) tile = t;
    TL_REQUIRE(tile >= 0, "gemm_swiglu_direct: no tile of %d x %d with the fused gate", BM, BN);
    const int N = ((I + 31) / 32) * 64;
    const int rc = launch_dl_tile<bf16_t, true>((DlTile)tile, x, w, nullptr, 0, out, M, N, K, ldx, ldo, I, stream);
    if (rc != TL_OK) return rc;
    TL_CHECK_LAUNCH("gemm_dl_tile");
    return TL_OK;
}

// One tile shape with K split into `parts` (float slabs [parts, M, N]); for tests and tuning.
// stages == 4 with 128 x 128: the four-slab instance.
extern "C" int tl_gemm_direct_split_variant(const void* x, const void* w, void* out, int M, int N, int K, int ldx,
                                            int BM, int BN, int parts, int stages, hipStream_t stream) {
    TL_REQUIRE(M > 0 && K % 64 == 0 && ldx % 8 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0 && parts >= 1,
               "gemm_direct_split: needs M > 0, K a multiple of 64 and 16-byte aligned rows");
    int tile = -1;
    for (int t = 0; t < DL_TILES; ++t)
        if (DL_BM[t] == BM && DL_BN[t] == BN && (t == DL_128x128_S4) == (stages == 4)) tile = t;
    TL_REQUIRE(tile >= 0, "gemm_direct_split: no tile of %d x %d with %d stages", BM, BN, stages);
    const int steps = K / 64;
    const int k_per = ((steps + parts - 1) / parts) * 64;
    TL_REQUIRE((K + k_per - 1) / k_per == parts, "gemm_direct_split: %d parts leave one empty (K=%d)", parts, K);
    const int rc = launch_dl_tile<float, false>((DlTile)tile, x, w, nullptr, 0, out, M, N, K, ldx, N, 0, stream, parts, k_per);
    if (rc != TL_OK) return rc;
    TL_CHECK_LAUNCH("gemm_direct_split");
    return TL_OK;
}

static bool skinny_fits(const void* x, const void* w, int M, int K, int ldx) {
    return M <= 64 && K % 8 == 0 && ldx % 8 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0;
}

// out = x w^T (+ bias) in the engine's dtype: picks the kernel for the shape.
//   bfloat16, aligned, K a multiple of 64:
//     up to 64 rows as ring_pays says -> gemm_ring
//     one row against more, and up to 32 rows 2^23 numbers apart -> gemm_skinny (matrix cores, weight streaming)
//     everything else             -> gemm_dl_tile (matrix cores, operands straight into shared memory)
//   bfloat16, aligned, other K, M <= 64 -> gemm_skinny, except that 33..64 rows against a wide matrix go to the tile kernel
//   bfloat16, aligned, other K, M > 64  -> gemm_mfma_tile (matrix cores, shared-memory tiles)
//   32-bit, aligned, K a multiple of 32, M <= 16 as f32_few_rows_kernel says -> gemm_ring (true 32-bit arithmetic on the matrix cores)
//   32-bit, aligned, M <= 16    -> gemv_f32, above 8 rows gemv_f32_mfma (true 32-bit arithmetic, weight streaming)
//   32-bit, aligned, M > 16     -> gemm_f32_mfma (true 32-bit arithmetic on the matrix cores)
//   everything else             -> gemm_tile (true 32-bit arithmetic)
extern "C" int tl_gemm(const void* x, const void* w, const void* bias, int bias_f32, void* out,
                       int M, int N, int K, int ldx, int ldo, int dtype, int out_f32, hipStream_t stream) {
    TL_REQUIRE(M >= 0 && N > 0 && K > 0 && ldx >= K && ldo >= N, "gemm: bad sizes M=%d N=%d K=%d ldx=%d ldo=%d", M, N, K, ldx, ldo);
    if (M == 0) return TL_OK;
    const bool aligned = K % 8 == 0 && ldx % 8 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0;
    if (dtype == TL_DT_BF16 && ring_fits(x, w, M, K, ldx) && ring_pays(M, N, K)) {
        const RingCall c{x, w, bias, bias_f32, out, M, N, K, ldx, ldo, 0};
        return out_f32 ? launch_ring<float, 0, END_STORE>(c, stream) : launch_ring<bf16_t, 0, END_STORE>(c, stream);
    }
    if (dtype == TL_DT_BF16 && aligned && K % 64 == 0 && (M > 32 || (M > 8 && N >= 16384))) {      // (up to 32 rows of fewer columns: the rings', but for rows too far apart for their offsets and the tiles')
        int rc = out_f32 ? launch_dl_tile<float, false>(pick_dl_tile(M, N, K, false), x, w, bias, bias_f32, out, M, N, K, ldx, ldo, 0, stream)
                         : launch_dl_tile<bf16_t, false>(pick_dl_tile(M, N, K, false), x, w, bias, bias_f32, out, M, N, K, ldx, ldo, 0, stream);
        if (rc != TL_OK) return rc;
        TL_CHECK_LAUNCH("gemm_dl_tile");
        return TL_OK;
    }
    if (dtype == TL_DT_BF16 && aligned && (M > 64 || (M > 32 && N >= 16384))) {
        int rc;
        switch (pick_tile(M, N)) {
        case TILE_256x256: rc = launch_mfma_tile<256, 256, 4, 2, 64>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_f32, stream); break;
        case TILE_128x128_K32: rc = launch_mfma_tile<128, 128, 2, 2, 32>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_f32, stream); break;
        case TILE_128x128_K64: rc = launch_mfma_tile<128, 128, 2, 2, 64>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_f32, stream); break;
        default: rc = launch_mfma_tile<64, 128, 2, 2, 64>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_f32, stream); break;
        }
        if (rc != TL_OK) return rc;
        TL_CHECK_LAUNCH("gemm_mfma_tile");
        return TL_OK;
    }
    if (dtype == TL_DT_BF16 && skinny_fits(x, w, M, K, ldx)) {
        if (M <= 16) pick_skinny<1>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_f32, stream);
        else if (M <= 32) pick_skinny<2>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_f32, stream);
        else pick_skinny<4>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, out_f32, stream);
        TL_CHECK_LAUNCH("gemm_skinny");
        return TL_OK;
    }
    if (dtype == TL_DT_F32 && ring_fits_f32(x, w, M, K, ldx) && f32_few_rows_kernel(M, N, K) == 9) {
        const RingCall c{x, w, bias, bias_f32, out, M, N, K, ldx, ldo, 0};
        return launch_ring<float, 0, END_STORE, float>(c, stream);
    }
    if (dtype == TL_DT_F32 && gemv_f32_fits(x, w, M, K, ldx)) {
        if (M <= 8) launch_gemv_f32_fma<F32_PLAIN>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, F32Pairs{}, stream);
        else launch_gemv_f32_mfma(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, stream);
        TL_CHECK_LAUNCH("gemv_f32");
        return TL_OK;
    }
    if (dtype == TL_DT_F32 && gemm_f32_mfma_fits(x, w, M, K, ldx)) {
        launch_gemm_f32_mfma(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, stream);
        TL_CHECK_LAUNCH("gemm_f32_mfma");
        return TL_OK;
    }
    return tl_gemm_general(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, dtype, out_f32, stream);
}

// The fused query/key/value projection of up to 16 rows: out[:, :q_heads * head_dim] = rotated queries,
// rotated keys and values go to their pages (see RopeArgs; the weight rows of every query and key head
// are in the pair layout).  Returns TL_NOT_FUSED (nothing launched) for shapes it is not built for;
// the caller then runs the product and the rotation as two kernels.
#define TL_NOT_FUSED 100
template <int KS, bool XL, int R = 1>
static void launch_skinny_rope(const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int N, int K,
                               int ldx, int ldo, const RopeArgs& ra, hipStream_t stream, int rows_per_strip = 0) {
    const int rps = rows_per_strip > 0 ? rows_per_strip : 16 * R;
    dim3 grid((N + rps - 1) / rps), block(KS * 64);
    const size_t lds = (size_t)KS * R * 1024 + (XL ? (size_t)M * (K + 8) * 2 : 0);
    auto kernel = gemm_skinny_kernel<R, 1, KS, bf16_t, false, XL, 2, true>;
    if (XL) { static hipError_t allowed = allow_lds(kernel, 96 * 1024); (void)allowed; }
    kernel<<<grid, block, lds, stream>>>((const bf16_t*)x, (const bf16_t*)w, bias, bias_f32, (bf16_t*)out, M, N, K, ldx, ldo, 0, 0, rps, 0, ra, NormArgs{}, GroupStride{});
}

extern "C" int tl_gemm_partials_pay(int M, int N, int K);

extern "C" int tl_gemm_rope(const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int N, int K,
                            int ldx, int ldo, const void* positions, const void* inv_freq, const void* token_req,
                            const void* block_table, int bt_stride, void* k_plane, void* v_plane, int page,
                            int q_heads, int kv_heads, int head_dim, hipStream_t stream) {
    TL_REQUIRE(M > 0 && N > 0 && K > 0 && ldx >= K && ldo >= q_heads * head_dim, "gemm_rope: bad sizes M=%d N=%d K=%d", M, N, K);
    TL_REQUIRE(positions && inv_freq && head_dim % 4 == 0 && q_heads >= 0 && kv_heads >= 0, "gemm_rope: needs positions, frequencies and a head size that is a multiple of 4");
    TL_REQUIRE((k_plane == nullptr) == (v_plane == nullptr) && (!k_plane || (token_req && block_table && page > 0 && bt_stride > 0)),
               "gemm_rope: the cache write needs both planes, the block table and the requests of the rows");
    TL_REQUIRE(N == (q_heads + (k_plane ? 2 * kv_heads : 0)) * head_dim, "gemm_rope: %d output columns do not match the heads", N);
    const int strips = (N + 15) / 16, ks = strips >= 1024 ? 16 : 8;
    const bool rings = ring_fits(x, w, M, K, ldx) && ks == 8;      // (ks 16: as tl_gemm_rope_normed sums there)
    // (from 9 rows on the product split over K plus the rotation kernel that adds its slabs up stands beside it where that split is to be had)
    if (M > 16 || (M > 8 && tl_gemm_partials_pay(M, N, K)) || !skinny_fits(x, w, M, K, ldx) || N % 16 || ldo % 4 || ((uintptr_t)out % 8) || (!rings && K / 64 / ks >= 16) ||
        (k_plane && (((uintptr_t)k_plane % 8) || head_dim % 4)))
        return TL_NOT_FUSED;
    RopeArgs ra;
    ra.positions = (const int*)positions; ra.inv_freq = (const float*)inv_freq; ra.token_req = (const int*)token_req;
    ra.block_table = (const int*)block_table; ra.k_plane = (bf16_t*)k_plane; ra.v_plane = (bf16_t*)v_plane;
    ra.bt_stride = bt_stride; ra.page = page > 0 ? page : 1; ra.q_heads = q_heads; ra.kv_heads = k_plane ? kv_heads : 0; ra.head_dim = head_dim;
    if (rings) {
        RingCall c{x, w, bias, bias_f32, out, M, N, K, ldx, ldo, 0};
        c.ra = ra;
        return launch_ring<bf16_t, 0, END_ROTATE>(c, stream);
    }
    const bool xl = M > 1 && (size_t)M * (K + 8) * 2 <= SKINNY_XL_MAX_BYTES;
    int blocks = 1;
    const int rows = ks == 8 ? balanced_rows(N, &blocks) : 0;
    if (rows > 0 && blocks == 2) { if (xl) launch_skinny_rope<8, true, 2>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, ra, stream, rows); else launch_skinny_rope<8, false, 2>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, ra, stream, rows); }
    else if (ks == 8) { if (xl) launch_skinny_rope<8, true>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, ra, stream, rows); else launch_skinny_rope<8, false>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, ra, stream, rows); }
    else { if (xl) launch_skinny_rope<16, true>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, ra, stream); else launch_skinny_rope<16, false>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, ra, stream); }
    TL_CHECK_LAUNCH("gemm_rope");
    return TL_OK;
}

// What a fused norm needs to be right: whole 16-byte pieces everywhere, two pieces per thread at most.
static bool norm_fits(const NormArgs& na, int K, int threads) {
    return K % 8 == 0 && K <= 16 * threads && na.residual && na.residual_out && na.residual != na.residual_out && na.weight &&
           ((uintptr_t)na.residual % 16) == 0 && ((uintptr_t)na.residual_out % 16) == 0 && ((uintptr_t)na.weight % 16) == 0 &&
           ((uintptr_t)na.pending % 16) == 0 && (na.parts == 0 || na.part_stride % 4 == 0) && na.parts >= 0 && na.parts <= 64;
}

static NormArgs norm_args(const void* residual, void* residual_out, const void* pending, int parts, long part_stride,
                          const void* weight, int weight_f32, float eps) {
    NormArgs na;
    na.residual = (const float*)residual; na.residual_out = (float*)residual_out; na.pending = pending;
    na.weight = weight; na.part_stride = (size_t)part_stride; na.parts = parts; na.weight_f32 = weight_f32; na.eps = eps; na.share = na.strips = na.shares = 0;
    return na;
}

// The work-groups of a projection of one row that keeps the order of gemm_ring_kernel's, whose work-groups have `share` outputs each: up to two to a compute unit, for as many shares each.  Returns
// the outputs of a strip (see equal_strips).
static int keep_shares(NormArgs& na, int share, int total) {
    const int rows = equal_strips(share, 32, true), count = (total + share - 1) / share;
    na.share = share;
    na.strips = (share + rows - 1) / rows;
    na.shares = (count + 2 * TL_COMPUTE_UNITS - 1) / (2 * TL_COMPUTE_UNITS);
    return rows;
}

// out[m, n] = act((x w^T)[m, n]) * table[ids[m], n] of up to 16 rows in bfloat16, the product and what follows in float (a row whose id is no row of the table keeps what it
// holds).  Returns TL_NOT_FUSED (nothing launched) for shapes it is not built for.
extern "C" int tl_gemm_token_gate(const void* x, const void* w, const void* ids, const void* table, int table_ld, int vocab, void* out, int M, int N, int K, int ldx, int ldo, int act,
                                  hipStream_t stream) {
    TL_REQUIRE(M > 0 && N > 0 && K > 0 && ldx >= K && ldo >= N && table_ld >= N && vocab > 0 && ids && table, "gemm_token_gate: bad sizes M=%d N=%d K=%d", M, N, K);
    TL_REQUIRE(known_activation(act) && !(act & ACT_PAIRS), "gemm_token_gate: unknown activation %d", act);
    if (M > 16 || !ring_fits(x, w, M, K, ldx) || !ring_pays(M, N, K)) return TL_NOT_FUSED;
    RingCall c{x, w, nullptr, 0, out, M, N, K, ldx, ldo, 0};
    c.tk = TokenRow{(const int*)ids, (const bf16_t*)table, table_ld, vocab, act};
    return launch_ring<bf16_t, 0, END_TOKEN>(c, stream);
}


// tl_gemm_rope for one row whose x is the norm of the residual stream, made inside the kernel (see NormArgs):
// pending is bfloat16 [K] (parts == 0), float [parts][part_stride] or null.  Returns TL_NOT_FUSED (nothing
// launched) for shapes it is not built for; the caller then runs the norm and tl_gemm_rope.
extern "C" int tl_gemm_rope_normed(const void* residual, void* residual_out, const void* pending, int parts, long part_stride,
                                   const void* norm_weight, int norm_weight_f32, float eps,
                                   const void* w, const void* bias, int bias_f32, void* out, int N, int K, int ldo,
                                   const void* positions, const void* inv_freq, const void* token_req,
                                   const void* block_table, int bt_stride, void* k_plane, void* v_plane, int page,
                                   int q_heads, int kv_heads, int head_dim, hipStream_t stream) {
    TL_REQUIRE(N > 0 && K > 0 && ldo >= q_heads * head_dim, "gemm_rope_normed: bad sizes N=%d K=%d", N, K);
    TL_REQUIRE(positions && inv_freq && head_dim % 4 == 0 && q_heads >= 0 && kv_heads >= 0, "gemm_rope_normed: needs positions, frequencies and a head size that is a multiple of 4");
    TL_REQUIRE((k_plane == nullptr) == (v_plane == nullptr) && (!k_plane || (token_req && block_table && page > 0 && bt_stride > 0)),
               "gemm_rope_normed: the cache write needs both planes, the block table and the request of the row");
    TL_REQUIRE(N == (q_heads + (k_plane ? 2 * kv_heads : 0)) * head_dim, "gemm_rope_normed: %d output columns do not match the heads", N);
    NormArgs na = norm_args(residual, residual_out, pending, parts, part_stride, norm_weight, norm_weight_f32, eps);
    const int strips = (N + 15) / 16, ks = strips >= 1024 ? 16 : 8;
    if (!norm_fits(na, K, ks * 64) || ((uintptr_t)w % 16) || N % 16 || ldo % 4 || ((uintptr_t)out % 8) || K / 64 / ks >= 16 ||
        (k_plane && (((uintptr_t)k_plane % 8) || head_dim % 4)))
        return TL_NOT_FUSED;
    RopeArgs ra;
    ra.positions = (const int*)positions; ra.inv_freq = (const float*)inv_freq; ra.token_req = (const int*)token_req;
    ra.block_table = (const int*)block_table; ra.k_plane = (bf16_t*)k_plane; ra.v_plane = (bf16_t*)v_plane;
    ra.bt_stride = bt_stride; ra.page = page > 0 ? page : 1; ra.q_heads = q_heads; ra.kv_heads = k_plane ? kv_heads : 0; ra.head_dim = head_dim;
    int blocks = 1;
    int rows = ks == 8 ? balanced_rows(N, &blocks) : 0, run = 0;
    if (ks == 8 && ring_spread(K)) {             // shares as tl_gemm_rope deals them (see ring_products), in equal strips of up to two blocks: the same bits, and with rows of weights a multiple of
                                                 // 4 KB apart the order is as good here (us, in step / turned: 2560 x 2048 7.1 / 7.2, 6144 x 4096 15.8 / 14.9, 10240 x 2048 18.9 / 15.8)
        rows = keep_shares(na, plan_ring(N, 1, 1, TL_COMPUTE_UNITS, true, true, false).rows, N);
        blocks = rows > 16 ? 2 : 1;
        run = na.shares * na.share;
    }
    dim3 grid(run > 0 ? (N + run - 1) / run : rows > 0 ? (N + rows - 1) / rows : strips);
    const size_t lds = (size_t)ks * blocks * 1024 + (size_t)(K + 8) * 2;
#define TL_NORMED_ROPE(R, TURN) gemm_skinny_kernel<R, 1, 8, bf16_t, false, true, 2, true, true, TURN><<<grid, dim3(8 * 64), lds, stream>>>( \
            nullptr, (const bf16_t*)w, bias, bias_f32, (bf16_t*)out, 1, N, K, K, ldo, 0, 0, rows, run, ra, na, GroupStride{})
    if (rows > 0 && blocks == 2) { if (run > 0) TL_NORMED_ROPE(2, true); else TL_NORMED_ROPE(2, false); }
    else if (ks == 8) { if (run > 0) TL_NORMED_ROPE(1, true); else TL_NORMED_ROPE(1, false); }
#undef TL_NORMED_ROPE
    else
        gemm_skinny_kernel<1, 1, 16, bf16_t, false, true, 2, true, true><<<grid, dim3(16 * 64), lds, stream>>>(
            nullptr, (const bf16_t*)w, bias, bias_f32, (bf16_t*)out, 1, N, K, K, ldo, 0, 0, 0, 0, ra, na, GroupStride{});
    TL_CHECK_LAUNCH("gemm_rope_normed");
    return TL_OK;
}

// tl_gemm_swiglu for one row whose x is the norm of the residual stream, made inside the kernel.  Returns
// TL_NOT_FUSED (nothing launched) for shapes it is not built for.
extern "C" int tl_gemm_swiglu_normed(const void* residual, void* residual_out, const void* pending, int parts, long part_stride,
                                     const void* norm_weight, int norm_weight_f32, float eps,
                                     const void* w, void* out, int I, int K, hipStream_t stream) {
    TL_REQUIRE(I > 0 && K > 0, "gemm_swiglu_normed: bad sizes I=%d K=%d", I, K);
    const NormArgs na = norm_args(residual, residual_out, pending, parts, part_stride, norm_weight, norm_weight_f32, eps);
    const int N = ((I + 31) / 32) * 64;          // rows of the interleaved matrix
    if (!norm_fits(na, K, 16 * 64) || ((uintptr_t)w % 16) || K / 64 / 16 >= 16)
        return TL_NOT_FUSED;
    const StripPlan p = plan_strips(I, 2 * TL_COMPUTE_UNITS, 16, false);       // every work-group makes x once and walks its run of outputs
    const size_t lds = (size_t)16 * 1024 + (size_t)(K + 8) * 2;
    gemm_skinny_kernel<1, 1, 16, bf16_t, true, true, 2, false, true><<<dim3(p.groups), dim3(16 * 64), lds, stream>>>(
        nullptr, (const bf16_t*)w, nullptr, 0, (bf16_t*)out, 1, N, K, K, I, I, 0, p.per_strip, p.per_group, RopeArgs{}, na, GroupStride{});
    TL_CHECK_LAUNCH("gemm_swiglu_normed");
    return TL_OK;
}

// out[M, I] = silu(x g^T) * (x u^T) for bfloat16, with w = the gate and up matrices interleaved
// in blocks of 32 rows (rows 64 b .. 64 b + 31: gate rows 32 b .., rows 64 b + 32 ..: the up rows
// of the same columns), padded with zero rows to a multiple of 64.  The gate is applied to the
// float accumulators, as the reference's fused kernel does
// (/root/reference/src/torchlet/v10_triton_paged_gqa/kernel/ffn_swiglu.py:139-160).
template <int GATE>
static int gemm_gated(const void* x, const void* w, void* out, int M, int I, int K, int ldx, int ldo, hipStream_t stream) {
    TL_REQUIRE(M >= 0 && I > 0 && K > 0 && ldx >= K && ldo >= I, "gemm_swiglu: bad sizes M=%d I=%d K=%d", M, I, K);
    TL_REQUIRE(K % 8 == 0 && ldx % 8 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0,
               "gemm_swiglu: needs K and the row stride of x to be multiples of 8 and 16-byte aligned operands");
    if (M == 0) return TL_OK;
    const int N = ((I + 31) / 32) * 64;          // rows of the interleaved matrix
    const bf16_t* xb = (const bf16_t*)x;
    const bf16_t* wb = (const bf16_t*)w;
    bf16_t* ob = (bf16_t*)out;
    if (ring_fits(x, w, M, K, ldx) && ring_pays_gated(M, I, K)) return launch_ring<bf16_t, GATE, END_STORE>(RingCall{x, w, nullptr, 0, out, M, N, K, ldx, ldo, I}, stream);
    if (M <= 16 || (M <= 32 && K % 64 != 0)) {
        if (M <= 16) launch_skinny_t<1, 1, 16, bf16_t, GATE>(xb, wb, nullptr, 0, ob, M, N, K, ldx, ldo, I, stream);
        else launch_skinny_t<1, 2, 16, bf16_t, GATE>(xb, wb, nullptr, 0, ob, M, N, K, ldx, ldo, I, stream);
    } else if (K % 64 == 0) {
        const int rc = launch_dl_tile<bf16_t, GATE>(pick_dl_tile(M, N, K, true), xb, wb, nullptr, 0, ob, M, N, K, ldx, ldo, I, stream);
        if (rc != TL_OK) return rc;
    } else {
        int rc;
        switch (pick_tile(M, N)) {
        case TILE_256x256: rc = launch_mfma_tile_t<256, 256, 4, 2, bf16_t, GATE, 64>(xb, wb, nullptr, 0, ob, M, N, K, ldx, ldo, I, stream); break;
        case TILE_128x128_K32: rc = launch_mfma_tile_t<128, 128, 2, 2, bf16_t, GATE, 32>(xb, wb, nullptr, 0, ob, M, N, K, ldx, ldo, I, stream); break;
        case TILE_128x128_K64: rc = launch_mfma_tile_t<128, 128, 2, 2, bf16_t, GATE, 64>(xb, wb, nullptr, 0, ob, M, N, K, ldx, ldo, I, stream); break;
        default: rc = launch_mfma_tile_t<64, 128, 2, 2, bf16_t, GATE, 64>(xb, wb, nullptr, 0, ob, M, N, K, ldx, ldo, I, stream); break;
        }
        if (rc != TL_OK) return rc;
    }
    TL_CHECK_LAUNCH("gemm_swiglu");
    return TL_OK;
}

// `act`: the gate's activation, 0 silu, 1 relu, 2 the tanh form of gelu.
extern "C" int tl_gemm_swiglu(const void* x, const void* w, void* out, int M, int I, int K, int ldx, int ldo, int act, hipStream_t stream) {
    TL_REQUIRE(act >= 0 && act <= 2, "gemm_swiglu: unknown gate %d", act);
    if (act == 2) return gemm_gated<3>(x, w, out, M, I, K, ldx, ldo, stream);
    return act == 1 ? gemm_gated<2>(x, w, out, M, I, K, ldx, ldo, stream) : gemm_gated<1>(x, w, out, M, I, K, ldx, ldo, stream);
}

// A 32-bit product of up to 16 rows whose matrix's rows a gate or a rotation joins by pairs (through the rings, 4 rows, us, two launches / one: gate and up of 2 x 18944 x 3584 94 + 5 / 93,
// query, key and value 4608 x 3584 14.9 + 4.5 / 18.4): the rings where they are taken (offsets to a pair's second row in 32 bits), the multiply-add kernel up
// to 8 rows.  Returns TL_NOT_FUSED (nothing launched) for the rest.  wj (for tests and tuning) > 0: the rings in shapes of wj requests, `rows` pairs of them used; < 0: the rings as they would be dealt.
template <int END>
static int f32_pairs(const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int K, int ldx, int ldo, const F32Pairs& pa, int wj, int rows, hipStream_t stream) {
    const int N = 2 * pa.count;
    if (M > 16 || !gemv_f32_fits(x, w, M, K, ldx)) return TL_NOT_FUSED;
    const bool rings = ring_fits_f32(x, w, M, K, ldx) && ((size_t)pa.span + 256) * K * 4 < ((size_t)1 << 32);
    if (wj) TL_REQUIRE(rings && (wj < 0 || (wj <= 8 && rows > 0 && rows <= 4 * wj)), "gemm_f32: %d pairs do not fit %d requests, or sizes that the rings are not built for", rows, wj);
    if (wj || (rings && f32_few_rows_kernel(M, N, K) == 9)) {
        RingCall c{x, w, bias, bias_f32, out, M, N, K, ldx, ldo, pa.count};
        c.pa = pa;
        return launch_ring<float, END == F32_GATE ? 1 : 0, END == F32_GATE ? END_STORE : END_ROTATE, float>(c, stream, RingPlan{max(wj, 0), rows});
    }
    if (M > 8) return TL_NOT_FUSED;
    launch_gemv_f32_fma<END>(x, w, bias, bias_f32, out, M, N, K, ldx, ldo, pa, stream);
    TL_CHECK_LAUNCH("gemv_f32");
    return TL_OK;
}

// out[m, i] = act((x w^T)[m, i]) * (x w^T)[m, I + i] in 32 bits: w holds the gate's I rows, then the up rows.
extern "C" int tl_gemm_gate_f32(const void* x, const void* w, void* out, int M, int I, int K, int ldx, int ldo, int act, int wj, int rows, hipStream_t stream) {
    TL_REQUIRE(M > 0 && I > 0 && I < (1 << 30) && K > 0 && ldx >= K && ldo >= I && act >= 0 && act <= 2, "gemm_gate_f32: bad sizes M=%d I=%d K=%d or an unknown gate %d", M, I, K, act);
    F32Pairs pa{};
    pa.count = pa.span = I;
    pa.act = act;
    return f32_pairs<F32_GATE>(x, w, nullptr, 0, out, M, K, ldx, ldo, pa, wj, rows, stream);
}

// tl_gemm_rope in 32 bits: the rows of the heads as they are, frequency j turning the elements j and j + head_dim / 2.
extern "C" int tl_gemm_rope_f32(const void* x, const void* w, const void* bias, int bias_f32, void* out, int M, int N, int K, int ldx, int ldo, const void* positions, const void* inv_freq,
                                const void* token_req, const void* block_table, int bt_stride, void* k_plane, void* v_plane, int page, int q_heads, int kv_heads, int head_dim, int wj, int rows,
                                hipStream_t stream) {
    TL_REQUIRE(M > 0 && N > 0 && K > 0 && ldx >= K && ldo >= q_heads * head_dim, "gemm_rope_f32: bad sizes M=%d N=%d K=%d", M, N, K);
    TL_REQUIRE(positions && inv_freq && head_dim > 0 && head_dim % 2 == 0 && q_heads >= 0 && kv_heads >= 0, "gemm_rope_f32: needs positions, frequencies and an even head size");
    TL_REQUIRE((k_plane == nullptr) == (v_plane == nullptr) && (!k_plane || (token_req && block_table && page > 0 && bt_stride > 0 && kv_heads > 0)),
               "gemm_rope_f32: the cache write needs both planes, the block table and the requests of the rows");
    TL_REQUIRE(N == (q_heads + (k_plane ? 2 * kv_heads : 0)) * head_dim, "gemm_rope_f32: %d output columns do not match the heads", N);
    const F32Pairs pa{N / 2, head_dim / 2, 0, (const int*)positions, (const float*)inv_freq, (const int*)token_req, (const int*)block_table, (float*)k_plane, (float*)v_plane,
                      bt_stride, page > 0 ? page : 1, q_heads, k_plane ? kv_heads : 0};
    return f32_pairs<F32_ROTATE>(x, w, bias, bias_f32, out, M, K, ldx, ldo, pa, wj, rows, stream);
}

// out[P, M, N] (float) = partial sums of x w^T over P ranges of K, for a product with too few output
// tiles to fill the GPU (a narrow matrix against few rows): P work-groups per tile keep all compute
// units busy; whoever reads the slabs adds them up.  Returns P through `parts` (the caller sizes
// `out` for tl_gemm_partials_max()).  More than 64 rows: see plan_dl_split (measured at 512 rows:
// 3584 x 18944 147 -> 82 us, 5120 x 13824 179 -> 82 us, 5120 x 27648 348 -> 150 us, the norm's sum
// included).  Up to 64 rows, where it pays (see gives_few_row_slabs), the rings or the
// direct-load tile kernel with 64 x 64 tiles (see slabs_by_rings); for other K the skinny kernel
// with R = 4 strips per work-group, which share every x fetch.
extern "C" int tl_gemm_partials_max() { return 8; }

// Whether a product of up to 64 rows is given in slabs, K dealt to the work-groups of a narrow matrix: from 2 rows on, and for one row against more than 4096 columns on 256 units.  The line was drawn
// when its other side were the few-rows kernel's strips (3584 x 3584, 8 rows 9.1 / 7.5 us, 5120 x 27648, one row 70.8 / 53).  Between a whole product and slabs through the rings it would lie elsewhere
// (us with the norm that adds them up, whole / slabs: 2 rows, 3584 x 3584 10.4 / 11.2, 5120 x 5120 15.5 / 16.5, 4096 x 4096 11.1 / 12.9, 3584 x 18944 29.3 / 29.9, 2048 x 5632 10.2 / 10.1; 16 rows,
// 3584 x 3584 11.3 / 11.6, 4096 x 4096 11.9 / 13.7, 3584 x 18944 33.0 / 31.8; 32 rows, 3584 x 3584 13.0 / 12.6, 3584 x 18944 41 / 31; 64 rows 16.3 / 14.2 and 56 / 35), but what a consumer has read
// in 32 bits it goes on reading in 32 bits, and a whole product is rounded to bfloat16.
static bool gives_few_row_slabs(int M, int N, int K) {
    return K % 64 == 0 && (M >= 2 || N > 16 * TL_COMPUTE_UNITS);
}

// Whether a consumer that can add slabs up should ask for them instead of the whole product.
extern "C" int tl_gemm_partials_pay(int M, int N, int K);

// How many parts tl_gemm_partials would use.
extern "C" int tl_gemm_partials_parts(int M, int N, int K) {
    if (M > 64 && K % 64 == 0) {
        const int parts = plan_dl_split(M, N, K).parts;
        return parts > 0 ? parts : 1;
    }
    if (gives_few_row_slabs(M, N, K)) {
        const long tiles = (long)((M + 63) / 64) * ((N + 63) / 64);
        int P = (int)(TL_COMPUTE_UNITS / tiles);          // about one work-group per compute unit
        const int by_k = K / 512;                         // at least eight slabs of 64 per part
        if (P > by_k) P = by_k;
        if (P > 8) P = 8;
        return P < 1 ? 1 : P;
    }
    int P = (K + 63) / 64 / 32;                           // skinny kernel: at least 32 steps (2048 columns) per part
    if (P > 8) P = 8;
    return P < 1 ? 1 : P;
}

extern "C" int tl_gemm_partials_pay(int M, int N, int K) {
    if (M > 64 && K % 64 == 0) return gives_slabs(M, N, K);
    return gives_few_row_slabs(M, N, K) && tl_gemm_partials_parts(M, N, K) > 1;
}

// Whether those slabs come from the rings or from tiles of 64 x 64.  Up to 32 rows the rings (us, tiles / rings: 16 rows, 2048 x 2048 4.4 / 3.5, 4096 x 8192 17.9 / 13.5, 3584 x 18944 26.8 / 24.4).
// 33 to 64 rows, with K long enough: where their equal shares give a unit an eighth fewer weight rows than a tile has (64 rows, 6144 x 13824 0.86 of the tiles' time, 3584 x 8192 0.89), or where
// every unit has 64 on both sides and the rings' order is turned (4096 x 8192 0.88, 2048 x 16384, 48 rows, 0.90).  Otherwise a work-group draws as much either way, and tiles, whose waves read a
// row of x once for 64 columns, are ahead (64 rows, 3072 x 8192 14.9 / 16.2, 2048 x 11008 13.8 / 14.9, 5120 x 8192 21.5 / 22.9, 4096 x 4096 11.1 / 11.4).
static bool slabs_by_rings(int M, int N, int K, int parts, int k_per) {
    if (M <= 32) return true;
    if (K < 8192) return false;
    const bool every_unit = N % 64 == 0 && N / 64 * parts == TL_COMPUTE_UNITS, turned = ring_spread(K) && k_per >= 2048;      // (2048: eight slabs a wave)
    return (every_unit && turned) || plan_ring(N, M, 1, TL_COMPUTE_UNITS / parts, false, ring_spread(K), parts > 1).rows <= 56;
}

// The same for tests: 0 the rings, 2 tiles.
extern "C" int tl_gemm_slabs_choice(int M, int N, int K) {
    const int steps = (K + 63) / 64, P = tl_gemm_partials_parts(M, N, K), k_per = ((steps + P - 1) / P) * 64;
    return slabs_by_rings(M, N, K, (K + k_per - 1) / k_per, k_per) ? 0 : 2;
}

extern "C" int tl_gemm_partials(const void* x, const void* w, void* out, int M, int N, int K, int ldx, int* parts,
                                hipStream_t stream) {
    TL_REQUIRE(M > 0 && N > 0 && K > 0 && ldx >= K, "gemm_partials: bad sizes M=%d N=%d K=%d", M, N, K);
    TL_REQUIRE(K % 8 == 0 && ldx % 8 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0,
               "gemm_partials: needs K and the row stride of x to be multiples of 8 and 16-byte aligned operands");
    if (M > 64 && K % 64 == 0) {
        DlSplit plan = plan_dl_split(M, N, K);
        if (plan.parts == 0) plan = DlSplit{pick_dl_tile(M, N, K, false), 1, 0};
        *parts = plan.parts;
        const int rc = launch_dl_tile<float, false>(plan.tile, x, w, nullptr, 0, out, M, N, K, ldx, N, 0, stream, plan.parts, plan.k_per);
        if (rc != TL_OK) return rc;
        TL_CHECK_LAUNCH("gemm_partials");
        return TL_OK;
    }
    const int steps = (K + 63) / 64;
    int P = tl_gemm_partials_parts(M, N, K);
    const int k_per = ((steps + P - 1) / P) * 64;
    P = (K + k_per - 1) / k_per;
    *parts = P;
    if (gives_few_row_slabs(M, N, K) && ring_fits(x, w, M, K, ldx) && slabs_by_rings(M, N, K, P, k_per))
        return launch_ring<float, 0, END_STORE>(RingCall{x, w, nullptr, 0, out, M, N, K, ldx, N, 0, P, k_per}, stream);
    if (gives_few_row_slabs(M, N, K)) {
        auto kernel = gemm_dl_tile_kernel<64, 64, 2, 2, 4, float, false>;
        constexpr size_t lds = (size_t)4 * 128 * 64 * sizeof(bf16_t);
        static hipError_t allowed = allow_lds(kernel, lds);
        TL_REQUIRE(allowed == hipSuccess, "gemm_partials: cannot get %zu bytes of shared memory", lds);
        dim3 grid(((M + 63) / 64) * ((N + 63) / 64), P), block(256);
        kernel<<<grid, block, lds, stream>>>((const bf16_t*)x, (const bf16_t*)w, nullptr, 0, (float*)out, M, N, K, ldx, N, 0, k_per, GroupStride{});
        TL_CHECK_LAUNCH("gemm_partials");
        return TL_OK;
    }
    TL_REQUIRE(M <= 64, "gemm_partials: more than 64 rows need K to be a multiple of 64 (M=%d K=%d)", M, K);
    dim3 grid((N + 63) / 64, P), block(8 * 64);
    const size_t red_bytes = (size_t)8 * 4 * (M <= 16 ? 1 : (M <= 32 ? 2 : 4)) * 1024;
    if (M <= 16)
        gemm_skinny_kernel<4, 1, 8, float, false, false, skinny_depth<4, 1, 8>()><<<grid, block, red_bytes, stream>>>((const bf16_t*)x, (const bf16_t*)w, nullptr, 0, (float*)out, M, N, K, ldx, N, 0, k_per, 0, 0, RopeArgs{}, NormArgs{}, GroupStride{});
    else if (M <= 32)
        gemm_skinny_kernel<4, 2, 8, float, false, false, skinny_depth<4, 2, 8>()><<<grid, block, red_bytes, stream>>>((const bf16_t*)x, (const bf16_t*)w, nullptr, 0, (float*)out, M, N, K, ldx, N, 0, k_per, 0, 0, RopeArgs{}, NormArgs{}, GroupStride{});
    else {
        auto kernel = gemm_skinny_kernel<4, 4, 8, float, false, false, skinny_depth<4, 4, 8>()>;
        static hipError_t allowed = allow_lds(kernel, 128 * 1024);
        TL_REQUIRE(allowed == hipSuccess, "gemm_partials: cannot get %zu bytes of shared memory", red_bytes);
        kernel<<<grid, block, red_bytes, stream>>>((const bf16_t*)x, (const bf16_t*)w, nullptr, 0, (float*)out, M, N, K, ldx, N, 0, k_per, 0, 0, RopeArgs{}, NormArgs{}, GroupStride{});
    }
    TL_CHECK_LAUNCH("gemm_partials");
    return TL_OK;
}

// `groups` products of equal shape: out_g = x_g w_g^T with x_g = x + g * x_group (elements), w_g the g-th of the matrices [groups, N, K] and out_g =
// out + g * out_group.  One launch where the few-rows kernel or the direct-load tiles take the shape (bfloat16), one per product otherwise.
extern "C" int tl_gemm_groups(const void* x, long x_group, const void* w, void* out, long out_group, int groups, int M, int N, int K, int ldx, int ldo,
                              int dtype, int out_f32, hipStream_t stream) {
    TL_REQUIRE(groups > 0 && groups <= 64 && M >= 0 && N > 0 && K > 0 && ldx >= K && ldo >= N && x_group >= 0 && out_group >= 0, "gemm_groups: bad sizes groups=%d M=%d N=%d K=%d", groups, M, N, K);
    if (M == 0) return TL_OK;
    Groups gr;
    gr.count = groups;
    gr.stride = GroupStride{x_group, (long)N * K, out_group};
    const bool aligned = K % 8 == 0 && ldx % 8 == 0 && x_group % 8 == 0 && out_group % 8 == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0;
    if (dtype == TL_DT_BF16 && x_group % 8 == 0 && ring_fits(x, w, M, K, ldx) && ring_pays(M, (long)N * groups, K)) {
        RingCall c{x, w, nullptr, 0, out, M, N, K, ldx, ldo, 0};
        c.gr = gr;
        return out_f32 ? launch_ring<float, 0, END_STORE>(c, stream) : launch_ring<bf16_t, 0, END_STORE>(c, stream);
    }
    if (dtype == TL_DT_BF16 && aligned && K % 64 == 0 && (M > 32 || (M > 8 && (long)N * groups >= 16384))) {
        const DlTile tile = pick_dl_tile(M, N, K, false, groups);
        const int rc = out_f32 ? launch_dl_tile<float, false>(tile, x, w, nullptr, 0, out, M, N, K, ldx, ldo, 0, stream, 1, 0, gr)
                               : launch_dl_tile<bf16_t, false>(tile, x, w, nullptr, 0, out, M, N, K, ldx, ldo, 0, stream, 1, 0, gr);
        if (rc != TL_OK) return rc;
        TL_CHECK_LAUNCH("gemm_groups");
        return TL_OK;
    }
    if (dtype == TL_DT_BF16 && aligned && M <= 64) {
        if (M <= 16) pick_skinny<1>(x, w, nullptr, 0, out, M, N, K, ldx, ldo, out_f32, stream, gr);
        else if (M <= 32) pick_skinny<2>(x, w, nullptr, 0, out, M, N, K, ldx, ldo, out_f32, stream, gr);
        else pick_skinny<4>(x, w, nullptr, 0, out, M, N, K, ldx, ldo, out_f32, stream, gr);
        TL_CHECK_LAUNCH("gemm_groups");
        return TL_OK;
    }
    const size_t esize = dtype == TL_DT_BF16 ? 2 : 4, osize = (dtype == TL_DT_BF16 && !out_f32) ? 2 : 4;
    for (int g = 0; g < groups; ++g) {
        const int rc = tl_gemm((const char*)x + esize * g * x_group, (const char*)w + esize * g * N * K, nullptr, 0, (char*)out + osize * g * out_group, M, N, K,
                               ldx, ldo, dtype, out_f32, stream);
        if (rc != TL_OK) return rc;
    }
    return TL_OK;
}

// The same in bfloat16 for up to 16 rows, and beside them one more product of the same K: out2 [M, N2] (float) = x2 w2^T, rows of x2 ldx apart.  Returns TL_NOT_FUSED (nothing
// launched) for shapes it is not built for.
extern "C" int tl_gemm_groups_beside(const void* x, long x_group, const void* w, void* out, long out_group, int groups, int M, int N, int K, int ldx, int ldo, const void* x2,
                                     const void* w2, void* out2, int N2, hipStream_t stream) {
    TL_REQUIRE(groups > 0 && groups <= 64 && M > 0 && N > 0 && N2 > 0 && K > 0 && ldx >= K && ldo >= N && x_group >= 0 && out_group >= 0,
               "gemm_groups_beside: bad sizes groups=%d M=%d N=%d/%d K=%d", groups, M, N, N2, K);
    if (M > 16 || x_group % 8 || !ring_fits(x, w, M, K, ldx) || !ring_fits(x2, w2, M, K, ldx) || !ring_pays(M, (long)N * groups, K) || N2 > N) return TL_NOT_FUSED;
    RingCall c{x, w, nullptr, 0, out, M, N, K, ldx, ldo, 0};
    c.gr.count = groups;
    c.gr.stride = GroupStride{x_group, (long)N * K, out_group};
    c.be = Beside{(const bf16_t*)x2, (const bf16_t*)w2, (float*)out2, N2, groups};
    return launch_ring<bf16_t, 0, END_BESIDE>(c, stream);
}
