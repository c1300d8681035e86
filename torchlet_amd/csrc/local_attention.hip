// Attention over a paged cache whose keys and values differ in size (dim and vdim numbers per head), with soft-capped scores and a
// local mask: a query at position p reads the keys j <= p of its own chunk (j / chunk == p / chunk, chunks counted from position 0)
// and, with a window, j > p - window.  Scores, softmax and the weighted sum are float whatever the activation type.
//   k_plane [pages, kv_heads, page_size, dim], v_plane [pages, kv_heads, vdim, page_size] (the values of a page lie transposed, so
//   that eight neighbouring keys' values of one column are 16 bytes side by side, which is how the matrix cores want them); key j
//   of a request lies in slot j % page_size of page block_table[request][j / page_size].
// Two more mechanisms, each switched on by its operand.  A sink: the softmax's denominator also holds exp(sink[head]), which has neither
// key nor value and is not scaled.  Pooled blocks: beside a window of `window` tokens a query at position p reads one key and one
// value for every block of `pool` positions that lies wholly before its window, blocks 0 .. (p - window + 1) / pool - 1; block b's key
// and value are the means of the cached keys and values of the positions b * pool .. b * pool + pool - 1 and lie, as a token's would, in
// row b of planes of their own with a block table of their own (pool_blocks_kernel makes them when a step brings a block's last token).
// A third one: values that lie in the cache turned by their own positions; a head's output at position p is turned back by p.
// A fourth one: a gate per head; a token's output of head h is multiplied by sigmoid(gate[token, h]).
#include <limits.h>

#include "common.h"

// ------------------------------------------------------------------ cache write
// Token t's keys and values go to their page; what would go to page 0 (the sentinel of rows that belong to no request) is dropped.
template <typename T>
__global__ void kv_cache_write_kernel(const T* __restrict__ k, int k_ld, const T* __restrict__ v, int v_ld, int kv_heads, int dim, int vdim,
                                      const int* __restrict__ token_req, const int* __restrict__ positions, const int* __restrict__ block_table,
                                      int table_ld, int table_width, T* __restrict__ k_plane, T* __restrict__ v_plane, int pages, int page_size) {
    const int t = blockIdx.x;
    const int p = positions[t], block = p / page_size;
    if (p < 0 || block >= table_width) return;
    const int page = block_table[(size_t)token_req[t] * table_ld + block];
    if (page <= 0 || page >= pages) return;
    const int slot = p % page_size;
    for (int i = threadIdx.x; i < kv_heads * dim; i += blockDim.x) {
        const int g = i / dim, d = i % dim;
        k_plane[(((size_t)page * kv_heads + g) * page_size + slot) * dim + d] = k[(size_t)t * k_ld + i];
    }
    for (int i = threadIdx.x; i < kv_heads * vdim; i += blockDim.x) {
        const int g = i / vdim, d = i % vdim;
        v_plane[(((size_t)page * kv_heads + g) * vdim + d) * page_size + slot] = v[(size_t)t * v_ld + i];
    }
}

extern "C" int tl_kv_cache_write(const void* k, int k_ld, const void* v, int v_ld, int tokens, int kv_heads, int dim, int vdim,
                                 const void* token_req, const void* positions, const void* block_table, int table_ld, int table_width,
                                 void* k_plane, void* v_plane, int pages, int page_size, int dtype, hipStream_t stream) {
    TL_REQUIRE(tokens >= 0 && kv_heads > 0 && dim > 0 && vdim > 0 && page_size > 0 && pages > 0 && table_width > 0, "kv_cache_write: bad sizes");
    TL_REQUIRE(k_ld >= kv_heads * dim && v_ld >= kv_heads * vdim && table_ld >= table_width, "kv_cache_write: rows too short");
    if (tokens == 0) return TL_OK;
    if (dtype == TL_DT_F32)
        kv_cache_write_kernel<float><<<tokens, 256, 0, stream>>>((const float*)k, k_ld, (const float*)v, v_ld, kv_heads, dim, vdim, (const int*)token_req,
            (const int*)positions, (const int*)block_table, table_ld, table_width, (float*)k_plane, (float*)v_plane, pages, page_size);
    else if (dtype == TL_DT_BF16)
        kv_cache_write_kernel<bf16_t><<<tokens, 256, 0, stream>>>((const bf16_t*)k, k_ld, (const bf16_t*)v, v_ld, kv_heads, dim, vdim, (const int*)token_req,
            (const int*)positions, (const int*)block_table, table_ld, table_width, (bf16_t*)k_plane, (bf16_t*)v_plane, pages, page_size);
    else TL_REQUIRE(false, "kv_cache_write: unknown dtype %d", dtype);
    TL_CHECK_LAUNCH("kv_cache_write");
    return TL_OK;
}

// ------------------------------------------------------------------ the mask and the cap
struct LocalMask {
    int chunk, window;
    int keep_first;          // beside a window: the positions 0 .. keep_first - 1 are read by every later query, at their own places
    // the first key a query at position p reads
    __device__ __forceinline__ int first(int p) const {
        int lo = 0;
        if (chunk > 0) lo = max(lo, p / chunk * chunk);
        if (window > 0) lo = max(lo, p - window + 1);
        return lo;
    }
};

// The turn of a head's output back from its position (freq == null: none): of the first `dims` columns the pair (2m, 2m + 1), or, `halves`,
// (m, m + dims / 2), turns by -position * freq[m]; further columns pass.  Columns are taken in pairs, pair m at column_a(m) and column_b(m).
struct OutputTurn {
    const float* freq;       // [dims / 2]
    int dims, halves;
    __device__ __forceinline__ int column_a(int m) const { return (halves && m < dims / 2) ? m : 2 * m; }
    __device__ __forceinline__ int column_b(int m) const { return (halves && m < dims / 2) ? m + dims / 2 : 2 * m + 1; }
    __device__ __forceinline__ void turn(int m, int position, float& u, float& v) const {
        if (m >= dims / 2) return;
        float sn, c;
        sincosf((float)position * freq[m], &sn, &c);
        const float a = u, b = v;
        u = __fmaf_rn(a, c, __fmul_rn(b, sn));
        v = __fmaf_rn(b, c, -__fmul_rn(a, sn));
    }
};

__device__ __forceinline__ float cap_score(float s, float cap) { return cap > 0.f ? cap * tanhf(s / cap) : s; }

// ------------------------------------------------------------------ the general kernel
// One work-group of four waves per token and query head.  The keys lo .. p come in blocks of 64, dealt to the waves in turn (block b
// to wave b % 4: a matter of the position alone, so a token's result does not depend on the step it is in).  Within a block a lane
// owns a key: its score is the dot product with the query (kept in shared memory, scaled); the wave's running maximum and sum move on,
// and then a lane owns columns of the values: it adds p_j v_j over the block's keys, the weights read across the wave.  The four
// waves' states are joined in their order at the end.
#define LA_WAVES 4
#define LA_MAX_DIM 256
#define LA_COLS (LA_MAX_DIM / TL_WAVE)

template <typename T>
__global__ void __launch_bounds__(LA_WAVES * TL_WAVE)
local_attention_kernel(const T* __restrict__ q, int q_ld, T* __restrict__ out, int out_ld, const T* __restrict__ k_plane,
                       const T* __restrict__ v_plane, const int* __restrict__ block_table, int table_ld, const int* __restrict__ token_req,
                       const int* __restrict__ positions, int heads, int kv_heads, int dim, int vdim, int page_size, float scale, float cap,
                       LocalMask mask, float gain, const float* __restrict__ sink, const T* __restrict__ pk_plane, const T* __restrict__ pv_plane,
                       const int* __restrict__ pool_table, int pool_table_ld, int pool, OutputTurn back, const T* __restrict__ gate, int gate_ld) {
    __shared__ float sq[LA_MAX_DIM];
    __shared__ float sm[LA_WAVES], sl[LA_WAVES];
    __shared__ float sacc[LA_WAVES][LA_MAX_DIM];
    const int t = blockIdx.x, head = blockIdx.y;
    const int wave = threadIdx.x / TL_WAVE, lane = threadIdx.x % TL_WAVE;
    const int g = head / (heads / kv_heads);
    const int p = positions[t];
    const int lo = mask.first(p);
    const int* table = block_table + (size_t)token_req[t] * table_ld;
    const int* ptable = pool > 0 ? pool_table + (size_t)token_req[t] * pool_table_ld : nullptr;
    const int npool = (pool > 0 && mask.window > 0) ? max(0, p - mask.window + 1) / pool : 0;      // pooled blocks: keys 0 .. npool - 1 of this query
    for (int d = threadIdx.x; d < dim; d += blockDim.x) sq[d] = to_float(q[(size_t)t * q_ld + head * dim + d]) * scale;
    __syncthreads();

    float m = -INFINITY, l = 0.f;
    float acc[LA_COLS];
#pragma unroll
    for (int c = 0; c < LA_COLS; ++c) acc[c] = 0.f;
    const int nkept = min(mask.keep_first, lo);          // kept first tokens that lie before the window: keys npool .. npool + nkept - 1
    const int nkeys = npool + nkept + p - lo + 1;
    for (int b = wave; b * TL_WAVE < nkeys; b += LA_WAVES) {
        const int u = b * TL_WAVE + lane;                // pooled blocks first, then the kept first tokens, then the tokens lo .. p
        const bool ok = u < nkeys;
        float s = -INFINITY;
        const T* vr0 = v_plane;                          // the key's values: column c at vr0[c * page_size]
        if (ok) {
            const bool pooled = u < npool;
            const int j = pooled ? u : (u < npool + nkept ? u - npool : lo + u - npool - nkept);
            const int page = (pooled ? ptable : table)[j / page_size];
            const size_t at = (size_t)page * kv_heads + g;
            const int slot = j % page_size;
            const T* kr = (pooled ? pk_plane : k_plane) + (at * page_size + slot) * dim;
            vr0 = (pooled ? pv_plane : v_plane) + at * vdim * page_size + slot;
            float dot = 0.f;
            for (int d = 0; d < dim; ++d) dot = fmaf(sq[d], to_float(kr[d]), dot);
            s = cap_score(dot, cap);
        }
        const float m_new = fmaxf(m, wave_max(s));
        const float w = ok ? expf(s - m_new) : 0.f;
        const float keep = expf(m - m_new);            // (0 for the first block: m = -inf)
        l = l * keep + wave_sum(w);
        m = m_new;
#pragma unroll
        for (int c = 0; c < LA_COLS; ++c) acc[c] *= keep;
        const int nb = min(TL_WAVE, nkeys - b * TL_WAVE);
        const unsigned long long vaddr = (unsigned long long)(uintptr_t)vr0;
        for (int i = 0; i < nb; ++i) {
            const float wi = __shfl(w, i, TL_WAVE);
            const unsigned long long ai = ((unsigned long long)(unsigned)__shfl((int)(vaddr >> 32), i, TL_WAVE) << 32) | (unsigned)__shfl((int)vaddr, i, TL_WAVE);
            const T* vr = (const T*)(uintptr_t)ai;
#pragma unroll
            for (int c = 0; c < LA_COLS; ++c) {
                const int col = lane + c * TL_WAVE;
                if (col < vdim) acc[c] = fmaf(wi, to_float(vr[(size_t)col * page_size]), acc[c]);
            }
        }
    }
    if (lane == 0) { sm[wave] = m; sl[wave] = l; }
#pragma unroll
    for (int c = 0; c < LA_COLS; ++c) sacc[wave][lane + c * TL_WAVE] = acc[c];
    __syncthreads();
    if (wave == 0) {
        float top = sm[0];
        for (int w = 1; w < LA_WAVES; ++w) top = fmaxf(top, sm[w]);
        if (sink) top = fmaxf(top, sink[head]);
        float den = 0.f, f[LA_WAVES];
        for (int w = 0; w < LA_WAVES; ++w) {
            f[w] = sl[w] > 0.f ? expf(sm[w] - top) : 0.f;       // a wave without keys: no share
            den = fmaf(sl[w], f[w], den);
        }
        if (sink) den += expf(sink[head] - top);
        float norm = gain / den;
        if (gate) norm *= sigmoid(to_float(gate[(size_t)t * gate_ld + head]));
        auto joined = [&](int col) {
            float o = 0.f;
            for (int w = 0; w < LA_WAVES; ++w) o = fmaf(sacc[w][col], f[w], o);
            return o * norm;
        };
        T* orow = out + (size_t)t * out_ld + head * vdim;
        if (back.freq) {
            for (int m = lane; m < vdim / 2; m += TL_WAVE) {
                const int ca = back.column_a(m), cb = back.column_b(m);
                float u = joined(ca), v = joined(cb);
                back.turn(m, p, u, v);
                orow[ca] = from_float<T>(u);
                orow[cb] = from_float<T>(v);
            }
        } else {
            for (int col = lane; col < vdim; col += TL_WAVE) orow[col] = from_float<T>(joined(col));
        }
    }
}


// ------------------------------------------------------------------ the matrix-core kernel (bfloat16, prompts)
// One work-group of four waves per tile of 16 consecutive tokens of a request and query head.  The tile's keys come in steps of 32, dealt
// to the waves in turn (step i to wave i % 4: a matter of the positions alone), so that the longest tile of a step, whose time is the
// chain of its steps, takes a quarter of them per wave; the four waves' running maxima, sums and outputs are joined through shared
// memory at the end.  The operands do not pass through shared memory: with v_mfma_f32_16x16x32_bf16 the first
// operand's lane holds 8 neighbouring k of one row, which for keys (rows of K, k along dim), queries (rows of Q, k along dim) and
// transposed values (rows of V^T, k along the keys of a page) are 16 bytes side by side in memory.
//   scores, transposed: S^T[key][token] = K Q^T.  A lane ends up with one token (lane % 16) and four keys (rows 4 q .. 4 q + 3, q = lane / 16)
//   per product.  A step takes 32 keys in two products whose rows are keys base + 8 (r / 4) + r % 4 and that plus 4, so a lane holds
//   the keys base + 8 q .. 8 q + 7 of its token: exactly the 8 neighbouring k of the second operand of
//   O^T[column][token] += V^T[column][key] P^T[key][token], with no exchange between lanes.
// Cap, mask, running maximum and sum are per token, that is per lane, with the maximum and the final sum joined across the four
// lanes of a token.  Weights are rounded to bfloat16 for the second product; sums are float.
typedef __bf16 la_bf16x8 __attribute__((ext_vector_type(8)));
typedef float la_f32x4 __attribute__((ext_vector_type(4)));
union LaFrag {
    uint4 u;
    la_bf16x8 v;
    uint16_t e[8];
};
#define LAM_TOKENS 16
#define LAM_KEYS 32
#define LAM_WAVES 4
#define LAM_STRIDE (LAM_WAVES * LAM_KEYS)      // keys from one step of a wave to its next

// The hardware's own 2^x and 1 / x (about one unit in the last place each): a tile's time is these, eight scores to a lane and step.
#define LA_LOG2E 1.4426950408889634f

__device__ __forceinline__ float cap_score_fast(float s, float cap, float two_log2e_over_cap) {
    if (cap <= 0.f) return s;
    // cap * tanh(s / cap) with tanh(x) = 1 - 2 / (e^(2 x) + 1); beyond |x| = 15 it is +-1 to the last bit
    const float e = __builtin_amdgcn_exp2f(fminf(fmaxf(s * two_log2e_over_cap, -43.f), 43.f));
    return cap * (1.f - 2.f * __builtin_amdgcn_rcpf(e + 1.f));
}

// HEADS: every request brings one token; a tile's 16 columns are heads of one key/value head (chunks of up to 16) instead of tokens of one head, so the
// heads read their keys and values once, and with splits > 1 a tile's keys are dealt to that many work-groups, each of which leaves its sums for
// local_merge_kernel.  Splits are what one request needs: a work-group's CU fetches at most 64 bytes a clock, 2 MB of a head's keys and values at 4000
// tokens take it 14 us.
// FRESH (with HEADS): the token's own key and value come from the projection's rows, and the wave whose keys they are among puts them into their pages, so that a decode step needs no launch for that ahead
// (8 tokens of 4 heads of 128 and 128: 5.0 us): the step that holds the token's key takes it from there instead of from the page, and nobody else reads its place.
struct FreshRows {
    const bf16_t *k, *v;     // row t: token t's keys (kv_heads * dim) and values (kv_heads * vdim)
    int k_ld, v_ld, pages;
};
template <int DK, int DV, bool HEADS, bool FRESH>          // dim / 32 and vdim / 16
__global__ void __launch_bounds__(256)
local_attention_mfma_kernel(const bf16_t* __restrict__ q, int q_ld, bf16_t* __restrict__ out, int out_ld, const bf16_t* k_plane,
                            const bf16_t* v_plane, FreshRows fresh, const int* __restrict__ block_table, int table_ld, int table_width,
                            const int* __restrict__ req_indptr, const int* __restrict__ ctx_lens, const int* __restrict__ tile_req,
                            const int* __restrict__ tile_tok0, int heads, int kv_heads, int page_size, float scale, float cap,
                            LocalMask mask, float gain, const float* __restrict__ sink, const bf16_t* __restrict__ pk_plane,
                            const bf16_t* __restrict__ pv_plane, const int* __restrict__ pool_table, int pool_table_ld, int pool_table_width, int pool,
                            OutputTurn back, const bf16_t* __restrict__ gate, int gate_ld, int below, float* __restrict__ part_o,
                            float2* __restrict__ part_ml) {
    constexpr int dim = DK * 32, vdim = DV * 16;
    extern __shared__ float la_smem[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, kq = lane >> 4;
    const int group = heads / kv_heads, chunks = (group + 15) / 16;
    const int g = HEADS ? blockIdx.y / chunks : blockIdx.y / group;
    const int head0 = HEADS ? g * group + blockIdx.y % chunks * 16 : blockIdx.y;      // the head of the first column
    const int split = HEADS ? blockIdx.z : 0, splits = HEADS ? gridDim.z : 1;
    const int tile = blockIdx.x;
    const int req = tile_req ? tile_req[tile] : tile;
    const int first = req_indptr[req], n_new = req_indptr[req + 1] - first;
    const int tok0 = tile_tok0 ? tile_tok0[tile] : 0;
    const int n_tile = min(LAM_TOKENS, n_new - tok0);            // tokens of this tile
    if (n_tile <= 0 || n_new >= below) return;                   // (requests of `below` tokens or more are local_prompt_kernel's)
    const int n_cols = HEADS ? min(16, group - blockIdx.y % chunks * 16) : n_tile;
    const int p0 = ctx_lens[req] + tok0;                         // position of the tile's first token
    const int my_tok = HEADS ? 0 : min(li, n_cols - 1);          // (lanes beyond the tile's columns repeat its last one and store nothing)
    const int my_head = HEADS ? head0 + min(li, n_cols - 1) : head0;
    const int my_p = p0 + my_tok, my_lo = mask.first(my_p);
    const int* table = block_table + (size_t)req * table_ld;
    const float inv_cap = cap > 0.f ? 2.f * LA_LOG2E / cap : 0.f;
    const bool pow2 = (page_size & (page_size - 1)) == 0;
    const int page_shift = __ffs(page_size) - 1;
    auto page_of = [&](int key) { return pow2 ? key >> page_shift : key / page_size; };
    auto slot_of = [&](int key) { return pow2 ? key & (page_size - 1) : key % page_size; };

    LaFrag qf[DK];
    {
        const bf16_t* qrow = q + (size_t)(first + tok0 + my_tok) * q_ld + my_head * dim + 8 * kq;
#pragma unroll
        for (int s = 0; s < DK; ++s) qf[s].u = *(const uint4*)(qrow + 32 * s);
    }
    la_f32x4 acc[DV];
#pragma unroll
    for (int j = 0; j < DV; ++j) acc[j] = la_f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;

    const int p_last = p0 + n_tile - 1;
    const bf16_t* fresh_k = FRESH ? fresh.k + (size_t)(first + tok0) * fresh.k_ld + g * dim : nullptr;
    uint16_t fresh_v[FRESH ? DV : 1];                            // this lane's columns of the token's own values
    if constexpr (FRESH) {
        const bf16_t* row = fresh.v + (size_t)(first + tok0) * fresh.v_ld + g * vdim + li;
#pragma unroll
        for (int j = 0; j < DV; ++j) fresh_v[j] = row[16 * j].bits;
    }
    // rows of the two score products that this lane fetches: keys base + 8 (li / 4) + li % 4 (+ 4)
    const int krow = 8 * (li >> 2) + (li & 3);
    // One pass over a stretch of keys lo_valid .. hi_valid of planes kp / vp (the tokens of the tile's reach, or the pooled blocks before its
    // window), of which this lane's token reads my_first .. my_last.  The running maximum, sum and output carry over from pass to pass.
    // `own`: the stretch ends with the token itself.
    auto run = [&](const bf16_t* kp, const bf16_t* vp, const int* __restrict__ tbl, int tbl_width, int lo_valid, int hi_valid,
                   int my_first, int my_last, bool own) {
        const int base0 = lo_valid / LAM_KEYS * LAM_KEYS;
        const int mine = base0 + LAM_KEYS * (split * LAM_WAVES + wave), stride = splits * LAM_STRIDE;      // (key steps are dealt to the splits' waves in turn)
        if (mine > hi_valid) return;
        // The pages of up to 64 blocks of the request lie in a register across the wave (lane i: block tab_first + i) and are read from
        // there, so that no fetch waits for a look-up in memory; the window moves on every 64 blocks.
        int tab_first = page_of(mine);
        int tab_reg = tbl[min(tab_first + lane, tbl_width - 1)];
        auto page_at = [&](int key) { return __shfl(tab_reg, page_of(key) - tab_first, TL_WAVE); };
        // The keys and values of a step are fetched one step ahead, while the step before is worked on.
        LaFrag a0[DK], a1[DK], va[DV], vb[DV];
        auto fetch = [&](int base, LaFrag (&vf)[DV]) {
            if (page_of(base + LAM_KEYS - 1) - tab_first >= TL_WAVE) {            // (the same for every lane)
                tab_first = page_of(base);
                tab_reg = tbl[min(tab_first + lane, tbl_width - 1)];
            }
            // keys: rows base + krow and base + krow + 4 (clamped into what exists: masked below)
            const int key0 = max(min(base + krow, hi_valid), lo_valid), key1 = max(min(base + krow + 4, hi_valid), lo_valid);
            const bf16_t* k0 = kp + (((size_t)page_at(key0) * kv_heads + g) * page_size + slot_of(key0)) * dim + 8 * kq;
            const bf16_t* k1 = kp + (((size_t)page_at(key1) * kv_heads + g) * page_size + slot_of(key1)) * dim + 8 * kq;
            if (FRESH && own) {
                if (key0 == hi_valid) k0 = fresh_k + 8 * kq;
                if (key1 == hi_valid) k1 = fresh_k + 8 * kq;
            }
#pragma unroll
            for (int s = 0; s < DK; ++s) { a0[s].u = *(const uint4*)(k0 + 32 * s); a1[s].u = *(const uint4*)(k1 + 32 * s); }
            // values, transposed: row = column of the values, k = keys base + 8 kq .. + 7 (one page: page_size % 8 == 0)
            const int key = base + 8 * kq;
            const int kc = max(min(key, hi_valid), lo_valid);
            const bf16_t* vt = vp + (((size_t)page_at(kc) * kv_heads + g) * vdim + li) * page_size + slot_of(key);
#pragma unroll
            for (int j = 0; j < DV; ++j) vf[j].u = *(const uint4*)(vt + (size_t)16 * j * page_size);      // (never conditional: nothing waits for it here)
        };
        auto step = [&](int base, LaFrag (&vf)[DV], LaFrag (&vnext)[DV]) {
            // ---- scores of 32 keys
            la_f32x4 s0 = la_f32x4{0.f, 0.f, 0.f, 0.f}, s1 = la_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < DK; ++s) {
                s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[s].v, qf[s].v, s0, 0, 0, 0);
                s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[s].v, qf[s].v, s1, 0, 0, 0);
            }
            if (base + stride <= hi_valid) fetch(base + stride, vnext);
            // ---- cap, mask, running maximum (scores in units of log 2 from here on, so that the weights are plain powers of two)
            float sc[8];
            float mx = -INFINITY;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int key = base + 8 * kq + e;
                const float raw = (e < 4 ? s0[e] : s1[e - 4]) * scale;
                sc[e] = (key <= my_last && key >= my_first) ? cap_score_fast(raw, cap, inv_cap) * LA_LOG2E : -INFINITY;
                mx = fmaxf(mx, sc[e]);
            }
            mx = max_across_halves(max_across_rows(mx));
            const float m_new = fmaxf(m, mx);
            const float m_use = m_new == -INFINITY ? 0.f : m_new;   // a token that has seen no key yet
            const float keep = __builtin_amdgcn_exp2f(m - m_use);   // (0 while m is -inf)
            m = m_new;
            LaFrag pf;
            float psum = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float w = __builtin_amdgcn_exp2f(sc[e] - m_use);
                const bf16_t wb = from_float<bf16_t>(w);
                pf.e[e] = wb.bits;
                psum += to_float(wb);                               // the sum of what the second product sees
            }
            l = l * keep + psum;
            // places no token has written yet, or whose page is gone, may hold anything: their values count as zero (first and last steps only)
            const int vkey = base + 8 * kq;
            if (vkey + 7 > hi_valid || vkey < lo_valid) {
#pragma unroll
                for (int j = 0; j < DV; ++j)
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (vkey + e > hi_valid || vkey + e < lo_valid) vf[j].e[e] = 0;
            }
            if (FRESH && own && vkey <= hi_valid && vkey + 7 >= hi_valid) {
#pragma unroll
                for (int j = 0; j < DV; ++j)
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (vkey + e == hi_valid) vf[j].e[e] = fresh_v[j];
            }
            if (__any(keep != 1.f)) {                               // (the maxima settle after a tile's first steps)
#pragma unroll
                for (int j = 0; j < DV; ++j) { acc[j][0] *= keep; acc[j][1] *= keep; acc[j][2] *= keep; acc[j][3] *= keep; }
            }
#pragma unroll
            for (int j = 0; j < DV; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[j].v, pf.v, acc[j], 0, 0, 0);
        };
        fetch(mine, va);
        for (int base = mine; base <= hi_valid; base += 2 * stride) {
            step(base, va, vb);
            if (base + stride <= hi_valid) step(base + stride, vb, va);
        }
    };
    if (pool > 0 && mask.window > 0) {
        // the pooled blocks that lie wholly before a token's window: 0 .. (p - window + 1) / pool - 1; the tile's last token reads the most
        const int n_tile_blocks = max(0, p_last - mask.window + 1) / pool, n_my_blocks = max(0, my_p - mask.window + 1) / pool;
        if (n_tile_blocks > 0)
            run(pk_plane, pv_plane, pool_table + (size_t)req * pool_table_ld, pool_table_width, 0, n_tile_blocks - 1, 0, n_my_blocks - 1, false);
    }
    if (mask.keep_first > 0 && mask.window > 0) {
        // the kept first tokens that lie before a token's window: 0 .. min(keep_first, its window's start) - 1; the tile's last token reads the most
        const int n_tile_kept = min(mask.keep_first, mask.first(p_last)), n_my_kept = min(mask.keep_first, my_lo);
        if (n_tile_kept > 0) run(k_plane, v_plane, table, table_width, 0, n_tile_kept - 1, 0, n_my_kept - 1, false);
    }
    // the first token reads furthest back; pages before may be gone
    run(k_plane, v_plane, table, table_width, mask.first(p0), p_last, my_lo, my_p, true);
    if constexpr (FRESH) {
        // the wave that has walked the token's own key (of the first work-group of a head's chunks) leaves it and its value in their page; page 0, the sentinel of rows that belong to no request, is never written
        const int steps = p_last / LAM_KEYS - mask.first(p0) / LAM_KEYS;
        if (steps % (splits * LAM_WAVES) == split * LAM_WAVES + wave && blockIdx.y % chunks == 0 && page_of(p_last) < table_width) {
            const int page = table[page_of(p_last)], slot = slot_of(p_last);
            if (page > 0 && page < fresh.pages) {
                bf16_t* kd = const_cast<bf16_t*>(k_plane) + (((size_t)page * kv_heads + g) * page_size + slot) * dim;
                bf16_t* vd = const_cast<bf16_t*>(v_plane) + ((size_t)page * kv_heads + g) * vdim * page_size + slot;
                for (int d = lane; d < dim; d += TL_WAVE) kd[d] = fresh_k[d];
                if (kq == 0) {
#pragma unroll
                    for (int j = 0; j < DV; ++j) vd[(size_t)(16 * j + li) * page_size] = bf16_t{fresh_v[j]};
                }
            }
        }
    }
    l = sum_across_halves(sum_across_rows(l));
    // ---- the four waves' shares are joined: per token the maxima, the sums and the outputs, in the order of the waves
    float* sm_m = la_smem;                              // [4][16], in units of log 2
    float* sm_l = sm_m + LAM_WAVES * LAM_TOKENS;        // [4][16]
    float* sm_o = sm_l + LAM_WAVES * LAM_TOKENS;        // [4][16][vdim]
    if (kq == 0) { sm_m[wave * LAM_TOKENS + li] = m; sm_l[wave * LAM_TOKENS + li] = l; }
    // acc[j][v] = O[token li][column 16 j + 4 kq + v]
#pragma unroll
    for (int j = 0; j < DV; ++j)
        *(float4*)(sm_o + ((size_t)wave * LAM_TOKENS + li) * vdim + 16 * j + 4 * kq) = make_float4(acc[j][0], acc[j][1], acc[j][2], acc[j][3]);
    __syncthreads();
    if (HEADS && splits > 1) {
        // this work-group's share: maximum, sum and weighted sum of the values, not yet divided
        for (int idx = threadIdx.x; idx < n_cols * vdim; idx += blockDim.x) {
            const int c = idx / vdim, col = idx % vdim;
            float top = sm_m[c];
#pragma unroll
            for (int w = 1; w < LAM_WAVES; ++w) top = fmaxf(top, sm_m[w * LAM_TOKENS + c]);
            const float use = top == -INFINITY ? 0.f : top;      // (a share without keys: zeros)
            float den = 0.f, o = 0.f;
#pragma unroll
            for (int w = 0; w < LAM_WAVES; ++w) {
                const float f = __builtin_amdgcn_exp2f(sm_m[w * LAM_TOKENS + c] - use);
                den = fmaf(sm_l[w * LAM_TOKENS + c], f, den);
                o = fmaf(sm_o[((size_t)w * LAM_TOKENS + c) * vdim + col], f, o);
            }
            const size_t at = ((size_t)first * heads + head0 + c) * splits + split;
            part_o[at * vdim + col] = o;
            if (col == 0) part_ml[at] = make_float2(top, den);
        }
        return;
    }
    // columns ca and cb of a token or head (cb < 0: ca alone)
    auto joined = [&](int tok, int ca, int cb, float& u, float& v) {
        const int head = HEADS ? head0 + tok : head0;
        const float sink2 = sink ? sink[head] * LA_LOG2E : -INFINITY;       // in units of log 2, like the maxima
        float top = sm_m[tok];
#pragma unroll
        for (int w = 1; w < LAM_WAVES; ++w) top = fmaxf(top, sm_m[w * LAM_TOKENS + tok]);
        top = fmaxf(top, sink2);
        float den = __builtin_amdgcn_exp2f(sink2 - top);                    // (0 without a sink)
        u = v = 0.f;
#pragma unroll
        for (int w = 0; w < LAM_WAVES; ++w) {
            const float f = __builtin_amdgcn_exp2f(sm_m[w * LAM_TOKENS + tok] - top);        // (0 for a wave that saw no key of this token)
            den = fmaf(sm_l[w * LAM_TOKENS + tok], f, den);
            const float* o = sm_o + ((size_t)w * LAM_TOKENS + tok) * vdim;
            u = fmaf(o[ca], f, u);
            if (cb >= 0) v = fmaf(o[cb], f, v);
        }
        float norm = gain / den;
        if (gate) norm *= sigmoid(to_float(gate[(size_t)(first + tok0 + (HEADS ? 0 : tok)) * gate_ld + head]));
        u *= norm;
        v *= norm;
    };
    bf16_t* const orow0 = out + (size_t)(first + tok0) * out_ld + head0 * vdim;
    const size_t col_ld = HEADS ? vdim : out_ld;
    if (back.freq) {
        for (int idx = threadIdx.x; idx < n_cols * (vdim / 2); idx += blockDim.x) {
            const int tok = idx / (vdim / 2), m = idx % (vdim / 2);
            const int ca = back.column_a(m), cb = back.column_b(m);
            float u, v;
            joined(tok, ca, cb, u, v);
            back.turn(m, HEADS ? p0 : p0 + tok, u, v);
            orow0[tok * col_ld + ca] = from_float<bf16_t>(u);
            orow0[tok * col_ld + cb] = from_float<bf16_t>(v);
        }
        return;
    }
    for (int idx = threadIdx.x; idx < n_cols * vdim; idx += blockDim.x) {
        const int tok = idx / vdim, col = idx % vdim;
        float u, v;
        joined(tok, col, -1, u, v);
        orow0[tok * col_ld + col] = from_float<bf16_t>(u);
    }
}

// A token's head from the shares of its splits: weights exp(m_s - M), the sink's term, then what the tile kernel does as it stores.  Four waves per token and head, each on a run of
// neighbouring splits in their order, lanes over pairs of columns; the runs' sums meet in shared memory in their order.  One trip to memory is what it costs: a wave asks for all its
// shares (LA_RUN at most at a time) before the weights are worked out.  (One wave with a chain of eight shares at a time: 7.5 us for one token's 16 heads of 16 shares, so 4.6.)
#define LA_RUN 8
__global__ void __launch_bounds__(4 * TL_WAVE)
local_merge_kernel(const float* __restrict__ part_o, const float2* __restrict__ part_ml, bf16_t* __restrict__ out, int out_ld, const int* __restrict__ req_indptr,
                   const int* __restrict__ ctx_lens, const int* __restrict__ tile_req, int heads, int vdim, int splits, float gain, const float* __restrict__ sink,
                   OutputTurn back, const bf16_t* __restrict__ gate, int gate_ld) {
    __shared__ float2 sums[4][TL_WAVE];
    const int req = tile_req ? tile_req[blockIdx.x] : blockIdx.x, head = blockIdx.y, lane = threadIdx.x % TL_WAVE, wave = threadIdx.x / TL_WAVE;
    const int token = req_indptr[req];
    if (req_indptr[req + 1] <= token) return;
    const size_t at = ((size_t)token * heads + head) * splits;
    const int each = (splits + 3) / 4, s0 = wave * each, s1 = min(splits, s0 + each);
    const float2 ml = lane < splits ? part_ml[at + lane] : make_float2(-INFINITY, 0.f);
    const float sink2 = sink ? sink[head] * LA_LOG2E : -INFINITY;
    const float* po = part_o + at * vdim;
    bf16_t* o = out + (size_t)token * out_ld + (size_t)head * vdim;
    for (int base = 0; base < vdim / 2; base += TL_WAVE) {
        const int m = min(base + lane, vdim / 2 - 1);                   // (lanes beyond the last pair repeat it and store nothing)
        const int ca = back.freq ? back.column_a(m) : 2 * m, cb = back.freq ? back.column_b(m) : 2 * m + 1;
        float top = 0.f, f = 0.f, u = 0.f, v = 0.f;
        for (int r = 0; r < each; r += LA_RUN) {
            float pu[LA_RUN], pv[LA_RUN];
#pragma unroll
            for (int e = 0; e < LA_RUN; ++e)
                if (r + e < each) {
                    const size_t row = (size_t)min(s0 + r + e, splits - 1) * vdim;      // (beyond the run: fetched, not added)
                    pu[e] = po[row + ca];
                    pv[e] = po[row + cb];
                }
            if (r == 0) {
                top = fmaxf(wave_max(ml.x), sink2);
                f = __builtin_amdgcn_exp2f(ml.x - top);                 // (0 for a share without keys)
            }
#pragma unroll
            for (int e = 0; e < LA_RUN; ++e)
                if (s0 + r + e < s1) {
                    const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), s0 + r + e));
                    u = fmaf(w, pu[e], u);
                    v = fmaf(w, pv[e], v);
                }
        }
        sums[wave][lane] = make_float2(u, v);
        __syncthreads();
        const float den = wave_sum(ml.y * f) + __builtin_amdgcn_exp2f(sink2 - top);
        if (wave == 0 && base + lane < vdim / 2) {
            float norm = gain / den;
            if (gate) norm *= sigmoid(to_float(gate[(size_t)token * gate_ld + head]));
#pragma unroll
            for (int w = 1; w < 4; ++w) { u += sums[w][lane].x; v += sums[w][lane].y; }
            u *= norm;
            v *= norm;
            if (back.freq) back.turn(m, ctx_lens[req], u, v);
            o[ca] = from_float<bf16_t>(u);
            o[cb] = from_float<bf16_t>(v);
        }
        __syncthreads();
    }
}

template <int DK, int DV, bool HEADS = false, bool FRESH = false>
static void launch_local_mfma(const void* q, int q_ld, void* out, int out_ld, const void* k_plane, const void* v_plane, const void* block_table,
                              int table_ld, int table_width, const void* req_indptr, const void* ctx_lens, const void* tile_req,
                              const void* tile_tok0, int tiles, int heads, int kv_heads, int page_size, float scale, float cap, LocalMask mask,
                              float gain, const void* sink, const void* pk_plane, const void* pv_plane, const void* pool_table, int pool_table_ld,
                              int pool_table_width, int pool, OutputTurn back, const void* gate, int gate_ld, int below, hipStream_t stream, int splits = 1, void* part_o = nullptr,
                              void* part_ml = nullptr, FreshRows fresh = FreshRows{}) {
    const int group = heads / kv_heads;
    dim3 grid(tiles, HEADS ? kv_heads * ((group + 15) / 16) : heads, splits), block(LAM_WAVES * TL_WAVE);
    const size_t smem = sizeof(float) * LAM_WAVES * LAM_TOKENS * (2 + DV * 16);
    auto kernel = local_attention_mfma_kernel<DK, DV, HEADS, FRESH>;
    static bool raised = false;                      // (per instance of the template)
    if (smem > 48 * 1024 && !raised) {
        hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
        raised = true;
    }
    kernel<<<grid, block, smem, stream>>>((const bf16_t*)q, q_ld, (bf16_t*)out, out_ld, (const bf16_t*)k_plane, (const bf16_t*)v_plane, fresh,
        (const int*)block_table, table_ld, table_width, (const int*)req_indptr, (const int*)ctx_lens, (const int*)tile_req, (const int*)tile_tok0,
        heads, kv_heads, page_size, scale, cap, mask, gain, (const float*)sink, (const bf16_t*)pk_plane, (const bf16_t*)pv_plane, (const int*)pool_table,
        pool_table_ld, pool_table_width, pool, back, (const bf16_t*)gate, gate_ld, below, (float*)part_o, (float2*)part_ml);
}

// Whether the matrix-core kernel is built for these sizes.
extern "C" int tl_local_attention_mfma_fits(int dim, int vdim, int page_size) {
    const bool dk = dim == 32 || dim == 64 || dim == 96 || dim == 128 || dim == 192 || dim == 256;
    const bool dv = vdim > 0 && vdim % 16 == 0 && (vdim <= 128 || vdim == 160 || vdim == 192 || vdim == 256);
    return dk && dv && page_size % 8 == 0;
}

// ------------------------------------------------------------------ long portions of prompts: 128 rows a work-group
// The same attention for requests that bring LP_LEAST tokens or more in a step that is large enough (local_prompt_pays).  A row is a token and one of up to gcap heads of a key/value
// head; four waves of 32 rows share steps of KEYS keys, which go from the pages straight into shared memory (STAGES steps of it, so that the next
// ones are on their way while this one is multiplied; 16-byte pieces whose slot in a row is exclusive-ored with the row against bank conflicts).
// Both products run transposed on v_mfma_f32_32x32x16_bf16: a lane owns one row (its maximum, sum and output), and the keys are dealt to the
// rows of the first product so that the weights a lane holds are the second product's operand as they stand (row 8 a + 4 h + b of a block of 32
// carries key 16 (a / 2) + 8 h + 4 (a % 2) + b).  The tile kernel above reads its operands from the caches for every 16 tokens of every head, and that
// traffic set its time; here 128 rows share them, and the matrix and vector units take turns at being the bound (0.77 PFLOP/s on long prompts).
// Measured against it, 32 heads of 128 over 8: a prompt of 4096 tokens 918 -> 178 us, 2048 305 -> 60, with a window of 512 181 -> 39; 64 heads of
// 192 / 128, 2048 tokens 817 -> 130.
// A tile takes up to three stretches of keys one after the other, each with limits of its own per row: the pooled blocks before the window, the
// kept first tokens, the tokens themselves.  Late tiles start first.
#define LP_ROWS 128
#define LP_BT_MAX 2048               // block-table entries of a stretch in shared memory
#define LP_LEAST 32                  // tokens of a request in a step
#define LP_HEADS_MOST 16             // heads of a tile
#define LP_DEEP 12.f                 // powers of two a step's reference may lie under the largest score so far (pages) ...
#define LP_SLACK 8.f                 // ... and a row's scores may rise above its reference before it is moved (rows side by side)

typedef float la_f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ void lp_load_to_lds(const void* base, unsigned offset, unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" :: "v"(offset), "s"(base), "s"(lds_addr) : "memory", "m0");
}

struct LocalArgs {
    const bf16_t* q;
    int q_ld;
    bf16_t* out;
    int out_ld;
    const bf16_t *k_plane, *v_plane;
    const int* block_table;
    int table_ld, table_width;
    const int *req_indptr, *ctx_lens;
    int requests, heads, kv_heads, gcap, page_size, page_shift;
    float scale, cap;
    LocalMask mask;
    float gain;
    const float* sink;
    const bf16_t *pk_plane, *pv_plane;
    const int* pool_table;
    int pool_table_ld, pool_table_width, pool;
    OutputTurn back;
    const bf16_t* gate;
    int gate_ld, least;
    // keys and values in rows side by side instead of pages (LINEAR): the i-th of `requests` portions is request portion_req[i]'s, whose key at
    // position p is row portion_at[i] + p - portion_low[i] (both multiples of 64); rows hold keys of all heads, k_ld numbers apart, then, from
    // shared_at bytes after k_plane, shared_ld numbers apart, the last dimensions of every head's key; values lie transposed, v_ld keys to a row
    const int *portion_req, *portion_at, *portion_low;
    int k_ld, shared_ld, v_ld;
    unsigned shared_at;
    const bf16_t* value_gate;            // every output number times the sigmoid of its own
    int value_gate_ld;
};

template <int DIM, int VDIM, int KEYS, int STAGES, bool CAP, bool LINEAR>
__global__ void __launch_bounds__(256, 2)
local_prompt_kernel(LocalArgs a) {
    constexpr int OWN = LINEAR && DIM > VDIM ? VDIM / 8 : DIM / 8;    // (LINEAR) pieces of a key row that are the head's own
    constexpr int KB = KEYS / 32, NC = DIM / 16, NB = VDIM / 32;      // blocks of keys; pieces of a score's sum; blocks of output columns
    constexpr int KPP = DIM / 8, VPP = KEYS / 8;                      // 16-byte pieces of a key row, of a row of transposed values
    constexpr int KBYTES = KEYS * DIM * 2, STAGE = KBYTES + VDIM * KEYS * 2;
    constexpr int KI = KBYTES / 4096, VI = VDIM * KEYS * 2 / 4096, NI = KI + VI;      // load instructions of a wave and step
    static_assert(KBYTES % 4096 == 0 && (VDIM * KEYS * 2) % 4096 == 0 && NI * (STAGES - 1) < 64, "whole instructions of four waves");
    extern __shared__ __attribute__((aligned(16))) unsigned char lp_smem[];
    int* bt = (int*)(lp_smem + STAGES * STAGE);
    const unsigned lds_base = (unsigned)(uintptr_t)((void __attribute__((address_space(3)))*)lp_smem);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 31, h = lane >> 5;
    auto key_slot = [](int piece, int key) { return DIM == 128 ? (piece ^ (key & 15)) : ((piece & ~7) | ((piece ^ (key >> 1)) & 7)); };
    auto value_slot = [](int piece, int d) { return KEYS == 64 ? (piece ^ ((d >> 1) & 7)) : (piece ^ ((d >> 2) & 3)); };

    // ---- which tile: the requests' tiles are counted by a prefix sum over the lanes; the last tile first, each with all its heads
    const int group = a.heads / a.kv_heads, chunks_h = (group + a.gcap - 1) / a.gcap, per_tile = a.kv_heads * chunks_h, tq = LP_ROWS / a.gcap;
    int total = 0;
    auto new_tokens = [&](int i) {
        if (i >= a.requests) return 0;
        const int r = LINEAR ? a.portion_req[i] : i;
        return a.req_indptr[r + 1] - a.req_indptr[r];
    };
    for (int base = 0; base < a.requests; base += TL_WAVE) {
        const int n = new_tokens(base + lane);
        int mine = n >= a.least ? (n + tq - 1) / tq : 0;
#pragma unroll
        for (int o = TL_WAVE / 2; o > 0; o >>= 1) mine += __shfl_xor(mine, o, TL_WAVE);
        total += __builtin_amdgcn_readfirstlane(mine);
    }
    if ((int)blockIdx.x >= total * per_tile) return;
    const int want = total - 1 - (int)blockIdx.x / per_tile, by = blockIdx.x % per_tile;
    int portion = 0, tok0 = 0;
    {
        int first = 0;
        for (int base = 0; base < a.requests; base += TL_WAVE) {
            const int n = new_tokens(base + lane);
            const int mine = n >= a.least ? (n + tq - 1) / tq : 0;
            int upto = mine;
#pragma unroll
            for (int o = 1; o < TL_WAVE; o <<= 1) {
                const int t = __shfl_up(upto, o, TL_WAVE);
                if (lane >= o) upto += t;
            }
            const unsigned long long past = __ballot(first + upto > want);
            if (past) {
                const int l = __builtin_amdgcn_readfirstlane(__ffsll(past) - 1);
                portion = base + l;
                tok0 = (want - first - __builtin_amdgcn_readlane(upto, l) + __builtin_amdgcn_readlane(mine, l)) * tq;
                break;
            }
            first += __builtin_amdgcn_readlane(upto, TL_WAVE - 1);
        }
    }
    const int g = by / chunks_h, g0 = by % chunks_h * a.gcap, gcount = min(a.gcap, group - g0);
    const int req = LINEAR ? __builtin_amdgcn_readfirstlane(a.portion_req[portion]) : portion;
    const int first = a.req_indptr[req], n_new = a.req_indptr[req + 1] - first, ctx = a.ctx_lens[req];
    const int ntok = min(tq, n_new - tok0), p0 = ctx + tok0, p_last = p0 + ntok - 1;

    const int row = wave * 32 + lr, r_tok = row / a.gcap, r_g = row % a.gcap;
    const bool row_ok = r_tok < ntok && r_g < gcount;
    const int r_pos = p0 + r_tok, r_head = g * group + g0 + r_g, r_token = first + tok0 + r_tok;
    const bool wave_has_rows = (wave * 32) / a.gcap < ntok;
    const int w_pos_min = p0 + min((wave * 32) / a.gcap, ntok - 1), w_pos_max = p0 + min((wave * 32 + 31) / a.gcap, ntok - 1);

    la_bf16x8 qf[NC];                        // my row's query: d = 16 c + 8 h .. + 7
    {
        const bf16_t* q = a.q + (size_t)r_token * a.q_ld + (size_t)r_head * DIM;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            LaFrag f;
            f.u = row_ok ? *(const uint4*)(q + 16 * c + 8 * h) : make_uint4(0, 0, 0, 0);
            qf[c] = f.v;
        }
    }
    // (waited for here, once: see the wait at a loop's head that the compiler would otherwise place)
#pragma unroll
    for (int c = 0; c < NC; ++c) asm volatile("" : "+v"(qf[c]));

    // what of a piece's address does not change from step to step: its key within the step, and bytes from the start of its page
    const int shift = a.page_shift, pmask = a.page_size - 1;
    unsigned k_off[KI], v_off[VI], k_step[LINEAR ? KI : 1];      // (LINEAR: bytes from one step's key to the next one's)
    int k_x[KI];
    int v_x;                                 // (the same in every value load of a lane: a piece's slot depends on the row's low bits alone)
#pragma unroll
    for (int j = 0; j < KI; ++j) {
        const int piece = (wave + 4 * j) * 64 + lane, kx = piece / KPP;
        k_x[j] = kx;
        const int slot = key_slot(piece % KPP, kx);
        if (LINEAR) {
            const bool own = slot < OWN;
            k_step[j] = (unsigned)(KEYS * (own ? a.k_ld : a.shared_ld)) * 2u;
            k_off[j] = own ? (unsigned)(kx * a.k_ld + g * (OWN * 8) + slot * 8) * 2u : a.shared_at + (unsigned)(kx * a.shared_ld + (slot - OWN) * 8) * 2u;
        } else k_off[j] = (unsigned)((g * a.page_size + (kx & pmask)) * DIM + slot * 8) * 2u;
    }
#pragma unroll
    for (int j = 0; j < VI; ++j) {
        const int piece = (wave + 4 * j) * 64 + lane, d = piece / VPP, x = 8 * value_slot(piece % VPP, d);
        if (j == 0) v_x = x;
        v_off[j] = LINEAR ? ((unsigned)(g * VDIM + d) * (unsigned)a.v_ld + (unsigned)x) * 2u : (unsigned)((g * VDIM + d) * a.page_size + (x & pmask)) * 2u;
    }
    const unsigned kpage = (unsigned)(a.kv_heads * a.page_size * DIM) * 2u, vpage = (unsigned)(a.kv_heads * a.page_size * VDIM) * 2u;
    const int krow = 16 * (lr >> 4) + 8 * ((lr >> 2) & 1) + 4 * ((lr >> 3) & 1) + (lr & 3);      // key that row lr of the first product carries

    // scores in units of log 2: with a cap they are capped first and then stand as they are, without one the factor goes into the exponent
    const float inv_cap = CAP ? 2.f * LA_LOG2E / a.cap : 0.f, scale2 = CAP ? 1.f : a.scale * LA_LOG2E;
    float m = -INFINITY, top = -INFINITY, l = 0.f;      // m: the reference of l and acc; top: the largest score so far (over pages)
    la_f32x16 acc[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[b][v] = 0.f;

    for (int phase = LINEAR ? 2 : 0; phase < 3; ++phase) {
        const bf16_t *kp = a.k_plane, *vp = a.v_plane;
        const int* tbl = LINEAR ? nullptr : a.block_table + (size_t)req * a.table_ld;
        int width = a.table_width, key_lo = 0, key_hi = 0;            // the tile reads keys key_lo .. key_hi - 1, ...
        int r_lo = 0, r_hi = -1, w_lo_max = 0, w_lo_min = 0, w_hi_min = -1, w_hi_max = -1;      // ... a row r_lo .. r_hi, and over the wave's rows
        if (phase == 0) {
            if (a.pool == 0 || a.mask.window == 0) continue;
            kp = a.pk_plane; vp = a.pv_plane;
            tbl = a.pool_table + (size_t)req * a.pool_table_ld;
            width = a.pool_table_width;
            auto blocks = [&](int p) { return max(0, p - a.mask.window + 1) / a.pool; };
            key_hi = blocks(p_last);
            r_hi = blocks(r_pos) - 1; w_hi_min = blocks(w_pos_min) - 1; w_hi_max = blocks(w_pos_max) - 1;
        } else if (phase == 1) {
            if (a.mask.keep_first == 0 || a.mask.window == 0) continue;
            auto kept = [&](int p) { return min(a.mask.keep_first, a.mask.first(p)); };
            key_hi = kept(p_last);
            r_hi = kept(r_pos) - 1; w_hi_min = kept(w_pos_min) - 1; w_hi_max = kept(w_pos_max) - 1;
        } else {
            key_lo = a.mask.first(p0);
            key_hi = p_last + 1;
            r_lo = a.mask.first(r_pos); r_hi = r_pos;
            w_lo_min = a.mask.first(w_pos_min); w_lo_max = a.mask.first(w_pos_max);
            w_hi_min = w_pos_min; w_hi_max = w_pos_max;
        }
        if (key_hi <= key_lo) continue;
        const int st_first = key_lo / KEYS, st_last = (key_hi + KEYS - 1) / KEYS;
        const int row0 = LINEAR ? a.portion_at[portion] - a.portion_low[portion] : 0;
        const int blk0 = (st_first * KEYS) >> shift, blk_n = ((key_hi - 1) >> shift) - blk0 + 1, blk_last = blk_n - 1;
        if (!LINEAR && (blk_n > LP_BT_MAX || blk0 + blk_n > width)) continue;      // (the host has seen to it that this cannot be)
        __syncthreads();                                              // the stretch before has been worked on
        if (!LINEAR) for (int i = threadIdx.x; i < blk_n; i += 256) bt[i] = tbl[max(blk0 + i, key_lo >> shift)];      // (pages before the first key may be gone)
        __syncthreads();
        int pg_k[KI], pg_v;
        auto look_up_one = [&](int st, int j) {
            if (LINEAR) return;
            const int first_key = st * KEYS - (blk0 << shift);
            if (j < KI) pg_k[j] = bt[min((first_key + k_x[j]) >> shift, blk_last)];
            else pg_v = bt[min((first_key + v_x) >> shift, blk_last)];
        };
        auto request_one = [&](int st, int buf, int j) {              // (after the step's look-ups)
            const unsigned sb = lds_base + buf * STAGE;
            if (LINEAR) {
                const unsigned at = (unsigned)(row0 + st * KEYS);
                if (j < KI) lp_load_to_lds(kp, at / KEYS * k_step[j] + k_off[j], sb + (wave + 4 * j) * 1024);
                else lp_load_to_lds(vp + at, v_off[j - KI], sb + KBYTES + (wave + 4 * (j - KI)) * 1024);
                return;
            }
            const unsigned uin = KEYS < a.page_size ? (unsigned)((st * KEYS) & pmask) : 0u;      // the step's first key's place in a longer page
            if (j < KI) lp_load_to_lds(kp + (size_t)uin * DIM, (unsigned)pg_k[j] * kpage + k_off[j], sb + (wave + 4 * j) * 1024);
            else lp_load_to_lds(vp + uin, (unsigned)pg_v * vpage + v_off[j - KI], sb + KBYTES + (wave + 4 * (j - KI)) * 1024);
        };
        auto look_up = [&](int st) {
#pragma unroll
            for (int j = 0; j <= KI; ++j) look_up_one(st, j);
        };
        // steps are requested STAGES - 1 ahead; past the end the last one again (nobody reads it), so that every wait is for the same count
#pragma unroll
        for (int i = 0; i < STAGES - 1; ++i) {
            const int st = min(st_first + i, st_last - 1);
            look_up(st);
#pragma unroll
            for (int j = 0; j < NI; ++j) request_one(st, i, j);
        }
        look_up(min(st_first + STAGES - 1, st_last - 1));
        asm volatile("s_waitcnt vmcnt(%0)" :: "n"(NI * (STAGES - 2)) : "memory");
        __syncthreads();
        for (int st = st_first; st < st_last; ++st) {
            const int buf = (st - st_first) % STAGES, buf_req = (st - st_first + STAGES - 1) % STAGES;
            const int st_req = min(st + STAGES - 1, st_last - 1), st_look = min(st + STAGES, st_last - 1), kbase = st * KEYS;
            unsigned char *kb_s = lp_smem + buf * STAGE, *vb_s = kb_s + KBYTES;
            if (!LINEAR && (kbase + KEYS > key_hi || kbase < key_lo)) {      // (LINEAR: such rows are zeros)
                // keys beyond the stretch's last may not be written yet, and the pages of those before its first may be gone: whatever lies there
                // must not reach the second product (0 * Inf), so their values count as zero
                for (int i = threadIdx.x; i < VDIM * VPP; i += 256) {
                    const int d = i / VPP, piece = i % VPP, k0 = kbase + 8 * piece;
                    if (k0 + 8 > key_hi || k0 < key_lo) {
                        LaFrag f;
                        uint4* ptr = (uint4*)(vb_s + d * (KEYS * 2) + value_slot(piece, d) * 16);
                        f.u = *ptr;
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            if (k0 + e >= key_hi || k0 + e < key_lo) f.e[e] = 0;
                        *ptr = f.u;
                    }
                }
                __syncthreads();
            }
            if (wave_has_rows && kbase <= w_hi_max && kbase + KEYS > w_lo_min) {
                la_f32x16 sc[KB];
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int v = 0; v < 16; ++v) sc[kb][v] = 0.f;
                constexpr int KAHEAD = 2;                 // a block's keys are read two products ahead
                LaFrag kf[KAHEAD + 1][KB];
                auto read_keys = [&](int c, int kb) {
                    const int kl = 32 * kb + krow;
                    kf[c % (KAHEAD + 1)][kb].u = *(const uint4*)(kb_s + kl * (DIM * 2) + key_slot(2 * c + h, kl) * 16);
                };
#pragma unroll
                for (int c = 0; c < KAHEAD; ++c)
#pragma unroll
                    for (int kb = 0; kb < KB; ++kb) read_keys(c, kb);
                __builtin_amdgcn_sched_barrier(0);
                constexpr int EVERY = NC * KB / NI;       // a request beside every so many products
                static_assert(EVERY >= 1, "a product for every request");
#pragma unroll
                for (int c = 0; c < NC; ++c)
#pragma unroll
                    for (int kb = 0; kb < KB; ++kb) {
                        sc[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[c % (KAHEAD + 1)][kb].v, qf[c], sc[kb], 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                        if (c + KAHEAD < NC) read_keys(c + KAHEAD, kb);
                        const int at = c * KB + kb;
                        if (at % EVERY == 0 && at / EVERY < NI) request_one(st_req, buf_req, at / EVERY);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                if (CAP) {
#pragma unroll
                    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                        for (int e = 0; e < 16; ++e) sc[kb][e] = cap_score_fast(sc[kb][e] * a.scale, a.cap, inv_cap) * LA_LOG2E;
                }
                float mloc = -INFINITY;
                if (kbase + KEYS - 1 <= w_hi_min && kbase >= w_lo_max) {
#pragma unroll
                    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                        for (int e = 0; e < 16; ++e) mloc = fmaxf(mloc, sc[kb][e]);
                } else {
#pragma unroll
                    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                        for (int e = 0; e < 16; ++e) {
                            const int key = kbase + 32 * kb + 16 * (e >> 3) + 8 * h + 4 * ((e >> 2) & 1) + (e & 3);
                            sc[kb][e] = (row_ok && key <= r_hi && key >= r_lo) ? sc[kb][e] : -INFINITY;
                            mloc = fmaxf(mloc, sc[kb][e]);
                        }
                }
                {
                    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(mloc), __float_as_uint(mloc), false, false);
                    mloc = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])) * scale2;
                }
                // The weights' rounding to bfloat16 is the largest error here, and it is least for those at and next below 1.  So over pages a step's weights are taken
                // from the step's own maximum (no more than LP_DEEP powers of two under the row's), and what stands in the sums is brought to that reference.  Error of
                // the output against 64 bits, 2048 tokens after 2000: 2.09e-3; 2.20e-3 in the tile kernel above, whose waves have a maximum each; 2.26e-3 with the row's
                // running maximum, and 2.34e-3 where the reference moves only when a row rises more than LP_SLACK above it, which takes 2 to 8 % less time.
                // Over rows of projected keys and values the last is enough, for there the rounding of the other operands counts as much: the mixer's error (16 heads of
                // 128 + 64 over 512 numbers, 512 / 2048 / 3001 tokens) is 5.34e-3 / 5.23e-3 / 5.15e-3, the absorbed way's 5.35e-3 / 5.31e-3 / 5.26e-3; the running maximum
                // takes 0.5 % off it and 8 % longer (4000 tokens in two portions, 93 -> 101 us each).
                if (!LINEAR) top = fmaxf(top, mloc);
                if (!LINEAR || __any(mloc > m + LP_SLACK)) {
                    const float m_new = LINEAR ? fmaxf(m, mloc) : fmaxf(mloc, top - LP_DEEP);
                    const float alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - m_new);
                    m = m_new;
                    l *= alpha;
#pragma unroll
                    for (int b = 0; b < NB; ++b) acc[b] *= alpha;
                }
                const float m_use = m == -INFINITY ? 0.f : -m;      // (nothing seen yet: every score is -inf)
                LaFrag pf[2 * KB];
                float psum = 0.f;
                auto weights = [&](int kb, int e0, int n) {
#pragma unroll
                    for (int e = e0; e < e0 + n; ++e) {
                        const __bf16 w = (__bf16)__builtin_amdgcn_exp2f(__builtin_fmaf(sc[kb][e], scale2, m_use));
                        psum += (float)w;                            // the sum of what the second product sees
                        pf[2 * kb + (e >> 3)].v[e & 7] = w;
                    }
                };
                // values: product i takes the columns 32 (i % NB) .. + 31 for the 16 keys of chunk i / NB, read two products ahead; the weights of a later
                // block and the next step's look-ups stand beside the products
                constexpr int NPV = 2 * KB * NB, VAHEAD = 2, PER = 16 / (2 * NB);
                LaFrag vf[VAHEAD + 1];
                auto read_values = [&](int i) {
                    const int d = 32 * (i % NB) + lr;
                    vf[i % (VAHEAD + 1)].u = *(const uint4*)(vb_s + d * (KEYS * 2) + value_slot(2 * (i / NB) + h, d) * 16);
                };
#pragma unroll
                for (int i = 0; i < VAHEAD; ++i) read_values(i);
                weights(0, 0, 16);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < NPV; ++i) {
                    acc[i % NB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i % (VAHEAD + 1)].v, pf[i / NB].v, acc[i % NB], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if (i + VAHEAD < NPV) read_values(i + VAHEAD);
                    const int kb = i / (2 * NB), within = i % (2 * NB);
                    if (kb + 1 < KB) weights(kb + 1, within * PER, PER);
                    else {
                        constexpr int LOOKS = (KI + 1 + 2 * NB - 1) / (2 * NB);
#pragma unroll
                        for (int u = 0; u < LOOKS; ++u)
                            if (within * LOOKS + u <= KI) look_up_one(st_look, within * LOOKS + u);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                l += psum;
            } else {
#pragma unroll
                for (int j = 0; j < NI; ++j) request_one(st_req, buf_req, j);
                look_up(st_look);
            }
            asm volatile("s_waitcnt vmcnt(%0)" :: "n"(NI * (STAGES - 2)) : "memory");
            __syncthreads();
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    l = sum_across_halves(l);
    if (!row_ok) return;
    // lane holds column 32 b + 8 q + 4 h + v of its row
    float norm = a.gain;
    if (a.sink) {
        const float sink2 = a.sink[r_head] * LA_LOG2E, top = fmaxf(m, sink2), keep = __builtin_amdgcn_exp2f(m - top);
        l = l * keep + __builtin_amdgcn_exp2f(sink2 - top);
        norm *= keep;
    }
    norm /= l;
    if (a.gate) norm *= sigmoid(to_float(a.gate[(size_t)r_token * a.gate_ld + r_head]));
    bf16_t* o = a.out + (size_t)r_token * a.out_ld + (size_t)r_head * VDIM;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int col = 32 * b + 8 * q + 4 * h;
            float y[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) y[v] = acc[b][4 * q + v] * norm;
            if (LINEAR && a.value_gate) {
                union { uint2 u; bf16_t e[4]; } vg;
                vg.u = *(const uint2*)(a.value_gate + (size_t)r_token * a.value_gate_ld + r_head * VDIM + col);
#pragma unroll
                for (int v = 0; v < 4; ++v) y[v] *= sigmoid(to_float(vg.e[v]));
            }
            if (!LINEAR && a.back.freq) {                // (pairs of neighbours: the host has seen to it)
                a.back.turn(col / 2, r_pos, y[0], y[1]);
                a.back.turn(col / 2 + 1, r_pos, y[2], y[3]);
            }
            union { uint2 u; uint16_t e[4]; } pk;
#pragma unroll
            for (int v = 0; v < 4; ++v) pk.e[v] = from_float<bf16_t>(y[v]).bits;
            *(uint2*)(o + col) = pk.u;
        }
}

// `tiles`: at most so many of LP_ROWS / gcap tokens (those beyond the last leave at once).
template <int DIM, int VDIM, int KEYS, int STAGES, bool CAP, bool LINEAR>
static int launch_local_prompt(const LocalArgs& a, long tiles, hipStream_t stream) {
    constexpr size_t smem = (size_t)STAGES * (KEYS * DIM * 2 + VDIM * KEYS * 2) + (LINEAR ? 0 : LP_BT_MAX * 4);
    auto kernel = local_prompt_kernel<DIM, VDIM, KEYS, STAGES, CAP, LINEAR>;
    static const hipError_t allowed = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (allowed != hipSuccess) { tl_set_error("local_prompt: cannot get %zu bytes of shared memory", smem); return TL_ERR_HIP; }
    const int group = a.heads / a.kv_heads;
    if (tiles > 0) kernel<<<dim3((unsigned)(tiles * a.kv_heads * ((group + a.gcap - 1) / a.gcap))), 256, smem, stream>>>(a);
    TL_CHECK_LAUNCH("local_prompt");
    return TL_OK;
}

// From where the kernel of 128 rows is the faster one: three of the tile kernel's work-groups (16 tokens of a head) to a CU.  That kernel deals a
// tile's keys to four waves and so fills the chip with few tokens already: with 32 heads over 8, 4000 cached tokens, 128 new ones take 55 us in it and
// 83 us here, 256 take 110 / 87, 512 take 206 / 98; 256 new ones beside 31 decoded tokens at 2000, where both kernels run, 189 / 207.  Tokens that
// must be decoded ones (all requests' but one each) do not count; a request of LP_LEAST tokens is where a step may hold no decoded ones at all
// (8 x 32 tokens of 64 heads after 1000: 94 / 54 us; below, most of a tile's rows would be empty).
static bool local_prompt_pays(const LocalArgs& a, long tokens) {
    const long more = tokens - a.requests + 1;
    return more >= LP_LEAST && more * a.heads >= 12288;
}

// Whether the kernel of 128 rows is built for these sizes: pages of a power of two of 8 keys or more, planes whose bytes 32 bits count, a request's
// blocks in its shared memory, a positive factor on the scores, outputs turned in neighbouring pairs.
static bool local_prompt_fits(const LocalArgs& a, int dim, int vdim, int pages, int pool_pages) {
    const bool sizes = (dim == 128 && vdim == 128) || (dim == 64 && vdim == 64) || (dim == 192 && vdim == 128);
    const long most = (long)(pages > pool_pages ? pages : pool_pages) * a.kv_heads * a.page_size * (dim > vdim ? dim : vdim) * 2;
    return sizes && a.page_size >= 8 && (a.page_size & (a.page_size - 1)) == 0 && most < (1L << 32) && a.table_width <= LP_BT_MAX &&
           a.pool_table_width <= LP_BT_MAX && a.scale > 0.f && !(a.back.freq && a.back.halves) && a.out_ld % 4 == 0 && ((uintptr_t)a.out % 8) == 0;
}

// Whether decoded tokens' heads go together (HEADS) at these sizes.
extern "C" int tl_local_heads_fits(int dim, int vdim) { return (dim == 64 || dim == 128 || dim == 192) && (vdim == 64 || vdim == 128); }

// Tiles of up to 16 consecutive tokens of one request: tile i belongs to request tile_req[i] (null: request i) and starts at that
// request's token tile_tok0[i] of the step (null: 0).  fresh_k, fresh_v (with splits; null: they are there): the tokens' own keys and values, which go to their pages.
extern "C" int tl_local_attention_tiles(const void* q, int q_ld, void* out, int out_ld, const void* k_plane, const void* v_plane, int pages,
                                        const void* block_table, int table_ld, int table_width, const void* req_indptr, const void* ctx_lens,
                                        const void* tile_req, const void* tile_tok0, int tiles, int heads, int kv_heads, int dim, int vdim,
                                        int page_size, float scale, float cap, int chunk, int window, float gain, const void* sink,
                                        const void* pk_plane, const void* pv_plane, const void* pool_table, int pool_table_ld, int pool_table_width,
                                        int pool, int keep_first, const void* turn_freq, int turn_dims, int turn_halves, const void* gate, int gate_ld,
                                        int tokens, int requests, int pool_pages, int splits, void* part_o, void* part_ml, const void* fresh_k, int fresh_k_ld, const void* fresh_v,
                                        int fresh_v_ld, hipStream_t stream) {
    TL_REQUIRE(!gate || gate_ld >= heads, "local_attention_tiles: a gate has a number per head");
    TL_REQUIRE(!turn_freq || (turn_dims > 0 && turn_dims % 2 == 0 && turn_dims <= vdim && vdim % 2 == 0), "local_attention_tiles: an output of %d columns turned over %d", vdim, turn_dims);
    TL_REQUIRE(keep_first >= 0 && (keep_first == 0 || (window > 0 && chunk == 0)), "local_attention_tiles: kept first tokens stand beside a window, without chunks");
    TL_REQUIRE(pool >= 0 && (pool == 0 || (window > 0 && pk_plane && pv_plane && pool_table && pool_table_ld >= pool_table_width && pool_table_width > 0)),
               "local_attention_tiles: pooled blocks need a window, their planes and their block table");
    TL_REQUIRE(tiles >= 0 && heads > 0 && heads <= 65535 && kv_heads > 0 && heads % kv_heads == 0 && page_size > 0, "local_attention_tiles: bad sizes");
    TL_REQUIRE(tl_local_attention_mfma_fits(dim, vdim, page_size), "local_attention_tiles: not built for heads of %d / %d numbers in pages of %d", dim, vdim, page_size);
    TL_REQUIRE(q_ld >= heads * dim && q_ld % 8 == 0 && ((uintptr_t)q & 15) == 0 && out_ld >= heads * vdim && table_ld >= table_width && chunk >= 0 && window >= 0,
               "local_attention_tiles: rows too short or not aligned");
    if (tiles == 0) return TL_OK;
    const LocalMask mask{chunk, window, keep_first};
    const OutputTurn back{(const float*)turn_freq, turn_dims, turn_halves};
    TL_REQUIRE(tokens >= 0 && requests >= 0 && pool_pages >= 0, "local_attention_tiles: bad sizes");
    const int group = heads / kv_heads, cut = (group + LP_HEADS_MOST - 1) / LP_HEADS_MOST;
    const LocalArgs a{(const bf16_t*)q, q_ld, (bf16_t*)out, out_ld, (const bf16_t*)k_plane, (const bf16_t*)v_plane, (const int*)block_table, table_ld,
                      table_width, (const int*)req_indptr, (const int*)ctx_lens, requests, heads, kv_heads, (group + cut - 1) / cut, page_size,
                      __builtin_ctz(page_size), scale, cap, mask, gain, (const float*)sink, (const bf16_t*)pk_plane, (const bf16_t*)pv_plane,
                      (const int*)pool_table, pool_table_ld, pool_table_width, pool, back, (const bf16_t*)gate, gate_ld, LP_LEAST, nullptr, nullptr, nullptr, 0, 0, 0, 0u, nullptr, 0};
    if (splits > 0) {        // one token a request, its heads together
        TL_REQUIRE(tl_local_heads_fits(dim, vdim) && tiles == tokens && splits <= TL_WAVE && (splits == 1 || (part_o && part_ml)), "local_attention_tiles: not built for these splits");
        TL_REQUIRE(!fresh_k || (fresh_v && !pool && fresh_k_ld >= kv_heads * dim && fresh_v_ld >= kv_heads * vdim && fresh_k_ld % 8 == 0 && ((uintptr_t)fresh_k & 15) == 0 && ((uintptr_t)fresh_v & 1) == 0),
                   "local_attention_tiles: the tokens' own keys lie in whole pieces, without pooled blocks");
        const FreshRows fresh{(const bf16_t*)fresh_k, (const bf16_t*)fresh_v, fresh_k_ld, fresh_v_ld, pages};
#define TL_LAH(DK, DV) if (fresh_k) TL_LAH_F(DK, DV, true); else TL_LAH_F(DK, DV, false)
#define TL_LAH_F(DK, DV, FRESH)                                                                                                              \
    launch_local_mfma<DK, DV, true, FRESH>(q, q_ld, out, out_ld, k_plane, v_plane, block_table, table_ld, table_width, req_indptr, ctx_lens,  \
                                    tile_req, tile_tok0, tiles, heads, kv_heads, page_size, scale, cap, mask, gain, sink, pk_plane, pv_plane, \
                                    pool_table, pool_table_ld, pool_table_width, pool, back, gate, gate_ld, INT_MAX, stream, splits, part_o, part_ml, fresh)
        if (dim == 64) { if (vdim == 64) { TL_LAH(2, 4); } else { TL_LAH(2, 8); } }
        else if (dim == 128) { if (vdim == 64) { TL_LAH(4, 4); } else { TL_LAH(4, 8); } }
        else { if (vdim == 64) { TL_LAH(6, 4); } else { TL_LAH(6, 8); } }
#undef TL_LAH_F
#undef TL_LAH
        TL_CHECK_LAUNCH("local_attention_heads");
        if (splits > 1) {
            local_merge_kernel<<<dim3(tiles, heads), 4 * TL_WAVE, 0, stream>>>((const float*)part_o, (const float2*)part_ml, (bf16_t*)out, out_ld, (const int*)req_indptr,
                (const int*)ctx_lens, (const int*)tile_req, heads, vdim, splits, gain, (const float*)sink, back, (const bf16_t*)gate, gate_ld);
            TL_CHECK_LAUNCH("local_merge");
        }
        return TL_OK;
    }
    TL_REQUIRE(!fresh_k, "local_attention_tiles: the tokens' own keys and values are written where a token's heads go together");
    int below = INT_MAX;
    if (tile_req && (long)tiles * LAM_TOKENS >= tokens && local_prompt_pays(a, tokens) && local_prompt_fits(a, dim, vdim, pages, pool_pages)) {
        const long most = tokens / LP_LEAST, tiles_most = tokens / (LP_ROWS / a.gcap) + (requests < most ? requests : most);
        int rc;
#define TL_LP(DIM, VDIM, KEYS, STAGES)                                                                        \
    rc = cap > 0.f ? launch_local_prompt<DIM, VDIM, KEYS, STAGES, true, false>(a, tiles_most, stream)         \
                   : launch_local_prompt<DIM, VDIM, KEYS, STAGES, false, false>(a, tiles_most, stream)
        if (dim == 192) TL_LP(192, 128, 32, 3); else if (dim == 128) TL_LP(128, 128, 64, 2); else TL_LP(64, 64, 64, 2);
#undef TL_LP
        if (rc != TL_OK) return rc;
        if (requests == 1 && (tiles - 1) * LAM_TOKENS + 1 >= LP_LEAST) return TL_OK;      // (its tiles show that it is a long one)
        below = LP_LEAST;
    }
#define TL_LAM(DK, DV)                                                                                                                      \
    launch_local_mfma<DK, DV>(q, q_ld, out, out_ld, k_plane, v_plane, block_table, table_ld, table_width, req_indptr, ctx_lens, tile_req,  \
                              tile_tok0, tiles, heads, kv_heads, page_size, scale, cap, mask, gain, sink, pk_plane, pv_plane, pool_table,        \
                              pool_table_ld, pool_table_width, pool, back, gate, gate_ld, below, stream)
#define TL_LAM_V(DK)                                     \
    switch (vdim) {                                      \
        case 16: TL_LAM(DK, 1); break;                   \
        case 32: TL_LAM(DK, 2); break;                   \
        case 48: TL_LAM(DK, 3); break;                   \
        case 64: TL_LAM(DK, 4); break;                   \
        case 80: TL_LAM(DK, 5); break;                   \
        case 96: TL_LAM(DK, 6); break;                   \
        case 112: TL_LAM(DK, 7); break;                  \
        case 128: TL_LAM(DK, 8); break;                  \
        case 160: TL_LAM(DK, 10); break;                 \
        case 192: TL_LAM(DK, 12); break;                 \
        default: TL_LAM(DK, 16); break;                  \
    }
    switch (dim) {
        case 32: TL_LAM_V(1) break;
        case 64: TL_LAM_V(2) break;
        case 96: TL_LAM_V(3) break;
        case 128: TL_LAM_V(4) break;
        case 192: TL_LAM_V(6) break;
        default: TL_LAM_V(8) break;
    }
#undef TL_LAM_V
#undef TL_LAM
    TL_CHECK_LAUNCH("local_attention_mfma");
    return TL_OK;
}

// ------------------------------------------------------------------ portions of prompts over rows of keys and values
// The kernel of 128 rows over keys and values that lie side by side for the step (LocalArgs: LINEAR), every head with keys and values of its own.  dim =
// own + shared numbers a key, own == vdim where a part is shared.  portion_* int32 [portions]; rows: of keys, a multiple of 64, zeros where no key is.
extern "C" int tl_prompt_rows_fits(int own, int shared, int vdim) {
    return (own == 128 && vdim == 128 && (shared == 0 || shared == 64)) || (own == 64 && vdim == 64 && shared == 0);
}

extern "C" int tl_prompt_rows(const void* q, int q_ld, void* out, int out_ld, const void* keys, int k_ld, long shared_at, int shared_ld, const void* values,
                              long rows, const void* portion_req, const void* portion_at, const void* portion_low, int portions, const void* req_indptr,
                              const void* ctx_lens, int tiles, int heads, int own, int shared, int vdim, float scale, int window, const void* sink,
                              const void* gate, int gate_ld, const void* value_gate, int value_gate_ld, hipStream_t stream) {
    TL_REQUIRE(tl_prompt_rows_fits(own, shared, vdim) && heads > 0 && scale > 0.f && window >= 0 && tiles >= 0 && portions >= 0, "prompt_rows: not built for these sizes");
    TL_REQUIRE(q_ld >= heads * (own + shared) && q_ld % 8 == 0 && ((uintptr_t)q & 15) == 0 && out_ld >= heads * vdim && out_ld % 4 == 0 && ((uintptr_t)out & 7) == 0,
               "prompt_rows: queries or output too short or not aligned");
    TL_REQUIRE(rows % 64 == 0 && k_ld >= heads * own && k_ld % 8 == 0 && ((uintptr_t)keys & 15) == 0 && ((uintptr_t)values & 15) == 0 &&
                   (shared == 0 || (shared_ld >= shared && shared_ld % 8 == 0 && shared_at % 16 == 0 && shared_at >= rows * k_ld * 2)),
               "prompt_rows: keys or values not aligned");
    TL_REQUIRE((shared ? shared_at + rows * shared_ld * 2 : rows * k_ld * 2) < (1L << 32) && rows * heads * vdim * 2 < (1L << 32), "prompt_rows: more keys than 32 bits count");
    TL_REQUIRE((!gate || gate_ld >= heads) && (!value_gate || (value_gate_ld >= heads * vdim && value_gate_ld % 4 == 0 && ((uintptr_t)value_gate & 7) == 0)),
               "prompt_rows: a gate that does not fit");
    if (tiles == 0 || portions == 0) return TL_OK;
    const LocalArgs a{(const bf16_t*)q, q_ld, (bf16_t*)out, out_ld, (const bf16_t*)keys, (const bf16_t*)values, nullptr, 0, 0, (const int*)req_indptr,
                      (const int*)ctx_lens, portions, heads, heads, 1, 64, 6, scale, 0.f, LocalMask{0, window, 0}, 1.f, (const float*)sink, nullptr, nullptr,
                      nullptr, 0, 0, 0, OutputTurn{nullptr, 0, 0}, (const bf16_t*)gate, gate_ld, 1, (const int*)portion_req, (const int*)portion_at,
                      (const int*)portion_low, k_ld, shared_ld, (int)rows, (unsigned)shared_at, (const bf16_t*)value_gate, value_gate_ld};
    if (shared) return launch_local_prompt<192, 128, 32, 3, false, true>(a, tiles, stream);
    return own == 128 ? launch_local_prompt<128, 128, 64, 2, false, true>(a, tiles, stream) : launch_local_prompt<64, 64, 64, 2, false, true>(a, tiles, stream);
}

extern "C" int tl_local_attention(const void* q, int q_ld, void* out, int out_ld, const void* k_plane, const void* v_plane, int pages,
                                  const void* block_table, int table_ld, int table_width, const void* token_req, const void* positions,
                                  int tokens, int heads, int kv_heads, int dim, int vdim, int page_size, float scale, float cap, int chunk,
                                  int window, float gain, const void* sink, const void* pk_plane, const void* pv_plane, const void* pool_table,
                                  int pool_table_ld, int pool, int keep_first, const void* turn_freq, int turn_dims, int turn_halves, const void* gate,
                                  int gate_ld, int dtype, hipStream_t stream) {
    TL_REQUIRE(!gate || gate_ld >= heads, "local_attention: a gate has a number per head");
    TL_REQUIRE(!turn_freq || (turn_dims > 0 && turn_dims % 2 == 0 && turn_dims <= vdim && vdim % 2 == 0), "local_attention: an output of %d columns turned over %d", vdim, turn_dims);
    TL_REQUIRE(keep_first >= 0 && (keep_first == 0 || (window > 0 && chunk == 0)), "local_attention: kept first tokens stand beside a window, without chunks");
    TL_REQUIRE(pool >= 0 && (pool == 0 || (window > 0 && pk_plane && pv_plane && pool_table)), "local_attention: pooled blocks need a window, their planes and their block table");
    TL_REQUIRE(tokens >= 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && vdim > 0 && page_size > 0, "local_attention: bad sizes");
    TL_REQUIRE(dim <= LA_MAX_DIM && vdim <= LA_MAX_DIM, "local_attention: built for heads of up to %d numbers, got %d / %d", LA_MAX_DIM, dim, vdim);
    TL_REQUIRE(q_ld >= heads * dim && out_ld >= heads * vdim && table_ld >= table_width && chunk >= 0 && window >= 0, "local_attention: rows too short");
    TL_REQUIRE(heads <= 65535, "local_attention: too many heads");
    if (tokens == 0) return TL_OK;
    const LocalMask mask{chunk, window, keep_first};
    const OutputTurn back{(const float*)turn_freq, turn_dims, turn_halves};
    dim3 grid(tokens, heads), block(LA_WAVES * TL_WAVE);
    if (dtype == TL_DT_F32)
        local_attention_kernel<float><<<grid, block, 0, stream>>>((const float*)q, q_ld, (float*)out, out_ld, (const float*)k_plane, (const float*)v_plane,
            (const int*)block_table, table_ld, (const int*)token_req, (const int*)positions, heads, kv_heads, dim, vdim, page_size, scale, cap, mask, gain,
            (const float*)sink, (const float*)pk_plane, (const float*)pv_plane, (const int*)pool_table, pool_table_ld, pool, back,
            (const float*)gate, gate_ld);
    else if (dtype == TL_DT_BF16)
        local_attention_kernel<bf16_t><<<grid, block, 0, stream>>>((const bf16_t*)q, q_ld, (bf16_t*)out, out_ld, (const bf16_t*)k_plane, (const bf16_t*)v_plane,
            (const int*)block_table, table_ld, (const int*)token_req, (const int*)positions, heads, kv_heads, dim, vdim, page_size, scale, cap, mask, gain,
            (const float*)sink, (const bf16_t*)pk_plane, (const bf16_t*)pv_plane, (const int*)pool_table, pool_table_ld, pool, back,
            (const bf16_t*)gate, gate_ld);
    else TL_REQUIRE(false, "local_attention: unknown dtype %d", dtype);
    TL_CHECK_LAUNCH("local_attention");
    return TL_OK;
}

// ------------------------------------------------------------------ pooled blocks
// Block b of a request (positions b * pool .. b * pool + pool - 1) gets its pooled key and value, the means of its cached keys and values,
// in the step that brings its last token: the blocks ctx / pool .. (ctx + n) / pool - 1 of a request that held ctx tokens and gets n.  One
// wave per such block, key/value head and 64 columns of keys-and-values side by side (a lane owns a column and walks the block's
// positions); sums in float in the order of the positions, one rounding.  Pooled rows lie in planes laid out like the tokens' (values
// transposed) under a block table of their own, block b in row b; what would go to page 0 is dropped.
template <typename T>
__global__ void __launch_bounds__(TL_WAVE)
pool_blocks_kernel(const T* __restrict__ k_plane, const T* __restrict__ v_plane, const int* __restrict__ block_table, int table_ld,
                   int table_width, T* __restrict__ pk_plane, T* __restrict__ pv_plane, const int* __restrict__ pool_table,
                   int pool_table_ld, int pool_table_width, const int* __restrict__ req_indptr, const int* __restrict__ ctx_lens,
                   int kv_heads, int dim, int vdim, int pages, int pool_pages, int page_size, int pool) {
    const int r = blockIdx.y;
    const int ctx = ctx_lens[r], n = req_indptr[r + 1] - req_indptr[r];
    const int b = ctx / pool + blockIdx.x;
    if (n <= 0 || b >= (ctx + n) / pool) return;
    const int pb = b / page_size;
    if (pb >= pool_table_width) return;
    const int ppage = pool_table[(size_t)r * pool_table_ld + pb];
    if (ppage <= 0 || ppage >= pool_pages) return;
    const int pslot = b % page_size;
    const int* table = block_table + (size_t)r * table_ld;
    const int chunks = (dim + vdim + TL_WAVE - 1) / TL_WAVE;
    const int g = blockIdx.z / chunks, e = (blockIdx.z % chunks) * TL_WAVE + threadIdx.x;
    if (e >= dim + vdim) return;
    const bool is_key = e < dim;
    const int d = is_key ? e : e - dim;
    // (sixteen positions' pages, then their numbers, are requested together: one after the other a block's 64 positions were a chain of 64 trips to memory: 2048 tokens, 4 heads 30.7 -> 13.3 us.  A
    // position without a page reads the sentinel's and is left out)
    constexpr int AHEAD = 16;
    float sum = 0.f;
    for (int j0 = 0; j0 < pool; j0 += AHEAD) {
        int at[AHEAD];
        T x[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int blk = (b * pool + j0 + u) / page_size;
            at[u] = j0 + u < pool && blk < table_width ? table[blk] : 0;
            if (at[u] < 0 || at[u] >= pages) at[u] = 0;
        }
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int slot = (b * pool + j0 + u) % page_size;
            x[u] = is_key ? k_plane[(((size_t)at[u] * kv_heads + g) * page_size + slot) * dim + d] : v_plane[(((size_t)at[u] * kv_heads + g) * vdim + d) * page_size + slot];
        }
#pragma unroll
        for (int u = 0; u < AHEAD; ++u)
            if (at[u] > 0) sum += to_float(x[u]);          // (a block's tokens are all held when its last one arrives)
    }
    const float mean = sum / (float)pool;
    if (is_key) pk_plane[(((size_t)ppage * kv_heads + g) * page_size + pslot) * dim + d] = from_float<T>(mean);
    else pv_plane[(((size_t)ppage * kv_heads + g) * vdim + d) * page_size + pslot] = from_float<T>(mean);
}

// `most_blocks`: an upper bound of the blocks one request completes in the step (its longest portion / pool + 1).
extern "C" int tl_pool_blocks(const void* k_plane, const void* v_plane, int pages, const void* block_table, int table_ld, int table_width,
                              void* pk_plane, void* pv_plane, int pool_pages, const void* pool_table, int pool_table_ld, int pool_table_width,
                              const void* req_indptr, const void* ctx_lens, int requests, int most_blocks, int kv_heads, int dim, int vdim,
                              int page_size, int pool, int dtype, hipStream_t stream) {
    TL_REQUIRE(requests >= 0 && requests <= 65535 && most_blocks >= 0 && kv_heads > 0 && dim > 0 && vdim > 0 && page_size > 0 && pool > 0 && pages > 0 && pool_pages > 0,
               "pool_blocks: bad sizes");
    TL_REQUIRE(table_ld >= table_width && pool_table_ld >= pool_table_width && table_width > 0 && pool_table_width > 0, "pool_blocks: block tables too short");
    if (requests == 0 || most_blocks == 0) return TL_OK;
    const int chunks = (dim + vdim + TL_WAVE - 1) / TL_WAVE;
    TL_REQUIRE((long)kv_heads * chunks <= 65535, "pool_blocks: too many heads");
    dim3 grid(most_blocks, requests, kv_heads * chunks), block(TL_WAVE);
    if (dtype == TL_DT_F32)
        pool_blocks_kernel<float><<<grid, block, 0, stream>>>((const float*)k_plane, (const float*)v_plane, (const int*)block_table, table_ld, table_width,
            (float*)pk_plane, (float*)pv_plane, (const int*)pool_table, pool_table_ld, pool_table_width, (const int*)req_indptr, (const int*)ctx_lens,
            kv_heads, dim, vdim, pages, pool_pages, page_size, pool);
    else if (dtype == TL_DT_BF16)
        pool_blocks_kernel<bf16_t><<<grid, block, 0, stream>>>((const bf16_t*)k_plane, (const bf16_t*)v_plane, (const int*)block_table, table_ld, table_width,
            (bf16_t*)pk_plane, (bf16_t*)pv_plane, (const int*)pool_table, pool_table_ld, pool_table_width, (const int*)req_indptr, (const int*)ctx_lens,
            kv_heads, dim, vdim, pages, pool_pages, page_size, pool);
    else TL_REQUIRE(false, "pool_blocks: unknown dtype %d", dtype);
    TL_CHECK_LAUNCH("pool_blocks");
    return TL_OK;
}

// ------------------------------------------------------------------ norm per head and rotation, in place
// x [T, ld] holds per token heads_a + heads_b heads of `dim` numbers side by side (queries, then keys).  One wave per token and head, in float:
//   norm (norm_a / norm_b != null): v <- v / sqrt(mean(v^2) + eps) * w[d], w = norm_a for the first heads_a heads, norm_b for the others;
//   without weights (`unit`): v <- v / sqrt(mean(v^2) + eps) for the heads of both kinds;
//   a temperature (`heat`) of the first heads_a heads (the queries): v <- v * (1 + coef * ln(floor((position + 1) / every) + 1));
//   rotation (inv_freq != null) of the first `dims` numbers by angle_i = float(position) * inv_freq[i]: pair (2i, 2i + 1), or, `halves`,
//   pair (i, i + dims / 2); (u, v) <- (u cos - v sin, v cos + u sin).  What lies beyond `dims` is not turned.  One rounding at the end.
// `raw_b` (optional, [T, raw_ld]): the heads_b heads as they come, before norm and rotation, are copied there (values that are the keys
// as projected).  `magnitude`: a factor on cosine and sine of these heads' rotation.
// `values`: heads_c more heads of vdim numbers behind those (the values), with a norm without a weight (`unit`) and a rotation of their own.
// `pages`: the heads_b and heads_c heads (keys and values) go to their pages instead of back to x, as kv_cache_write_kernel puts them there.
struct ValueHeads {
    int heads, vdim, unit;
    const float* inv_freq;
    int dims, halves;
};
struct QueryHeat {
    float coef;
    int every;                       // 0: none
};
template <typename T>
struct PagesOf {
    const int *token_req, *block_table;
    int table_ld, table_width;
    T *k_plane, *v_plane;            // null: x is written
    int pages, page_size;
};
#define HNR_WAVES 4
template <typename T>
__global__ void __launch_bounds__(HNR_WAVES * TL_WAVE)
head_norm_rotate_kernel(T* __restrict__ x, int ld, int tokens, int heads_a, int heads_b, int dim, const float* __restrict__ norm_a,
                        const float* __restrict__ norm_b, float eps, const int* __restrict__ positions, const float* __restrict__ inv_freq,
                        int dims, int halves, T* __restrict__ raw_b, int raw_ld, float magnitude, int unit, QueryHeat heat, ValueHeads values, PagesOf<T> to) {
    __shared__ float sv[HNR_WAVES][LA_MAX_DIM];
    const int wave = threadIdx.x / TL_WAVE, lane = threadIdx.x % TL_WAVE;
    const int heads_ab = heads_a + heads_b, heads = heads_ab + values.heads, keys_dim = dim;
    const long item = (long)blockIdx.x * HNR_WAVES + wave;
    const bool live = item < (long)tokens * heads;
    const int t = live ? (int)(item / heads) : 0, h = live ? (int)(item % heads) : 0;
    const bool is_value = h >= heads_ab;
    T* row = x + (size_t)t * ld + (is_value ? (size_t)heads_ab * dim + (size_t)(h - heads_ab) * values.vdim : (size_t)h * dim);
    float* v = sv[wave];
    const float* w = is_value ? nullptr : (h < heads_a ? norm_a : norm_b);
    const bool normed = is_value ? values.unit != 0 : (unit || w != nullptr);
    if (is_value) { dim = values.vdim; inv_freq = values.inv_freq; dims = values.dims; halves = values.halves; magnitude = 1.f; }
    float ss = 0.f;
    if (live) {
        T* raw = (raw_b && h >= heads_a && !is_value) ? raw_b + (size_t)t * raw_ld + (size_t)(h - heads_a) * dim : nullptr;
        for (int d = lane; d < dim; d += TL_WAVE) {
            const T x0 = row[d];
            if (raw) raw[d] = x0;
            const float a = to_float(x0); v[d] = a; ss = fmaf(a, a, ss);
        }
    }
    ss = wave_sum(ss);
    __syncthreads();
    if (live && normed) {
        const float inv = 1.f / sqrtf(ss / (float)dim + eps);
        for (int d = lane; d < dim; d += TL_WAVE) v[d] = v[d] * inv * (w ? w[d] : 1.f);
    }
    if (live && heat.every > 0 && h < heads_a) {         // (a lane goes over the numbers it normed itself)
        const float f = 1.f + heat.coef * logf((float)((positions[t] + 1) / heat.every + 1));
        for (int d = lane; d < dim; d += TL_WAVE) v[d] *= f;
    }
    __syncthreads();
    if (live && inv_freq) {
        const float pos = (float)positions[t];
        for (int i = lane; i < dims / 2; i += TL_WAVE) {
            const int ia = halves ? i : 2 * i, ib = halves ? i + dims / 2 : 2 * i + 1;
            float sn, c;
            sincosf(pos * inv_freq[i], &sn, &c);
            sn *= magnitude;
            c *= magnitude;
            const float a = v[ia], b = v[ib];
            v[ia] = __fmaf_rn(a, c, -__fmul_rn(b, sn));
            v[ib] = __fmaf_rn(b, c, __fmul_rn(a, sn));
        }
    }
    __syncthreads();
    if (!live) return;
    if (!to.k_plane || h < heads_a) {
        for (int d = lane; d < dim; d += TL_WAVE) row[d] = from_float<T>(v[d]);
        return;
    }
    const int p = positions[t], block = p / to.page_size;
    if (p < 0 || block >= to.table_width) return;
    const int page = to.block_table[(size_t)to.token_req[t] * to.table_ld + block];
    if (page <= 0 || page >= to.pages) return;          // page 0, the sentinel of rows that belong to no request, is never written
    const int at = p % to.page_size;
    if (is_value) {
        T* dst = to.v_plane + ((size_t)page * values.heads + h - heads_ab) * dim * to.page_size + at;
        for (int d = lane; d < dim; d += TL_WAVE) dst[(size_t)d * to.page_size] = from_float<T>(v[d]);
    } else {
        T* dst = to.k_plane + (((size_t)page * heads_b + h - heads_a) * to.page_size + at) * keys_dim;
        for (int d = lane; d < dim; d += TL_WAVE) dst[d] = from_float<T>(v[d]);
    }
}

extern "C" int tl_head_norm_rotate(void* x, int ld, int tokens, int heads_a, int heads_b, int dim, const void* norm_a, const void* norm_b, float eps,
                                   const void* positions, const void* inv_freq, int dims, int halves, void* raw_b, int raw_ld, float magnitude,
                                   int heads_c, int vdim, int unit_c, const void* inv_freq_c, int dims_c, int halves_c, const void* token_req,
                                   const void* block_table, int table_ld, int table_width, void* k_plane, void* v_plane, int pages, int page_size,
                                   int unit, float heat_coef, int heat_every, int dtype, hipStream_t stream) {
    TL_REQUIRE(!unit || (!norm_a && !norm_b), "head_norm_rotate: a norm has weights or it has none");
    TL_REQUIRE(heat_every >= 0 && (heat_every == 0 || positions), "head_norm_rotate: a temperature goes by positions");
    const QueryHeat heat{heat_coef, heat_every};
    TL_REQUIRE(heads_c >= 0 && (heads_c == 0 || (vdim > 0 && vdim <= LA_MAX_DIM && ld >= (heads_a + heads_b) * dim + heads_c * vdim)), "head_norm_rotate: bad sizes of the values");
    TL_REQUIRE(heads_c == 0 || !inv_freq_c || (positions && dims_c > 0 && dims_c % 2 == 0 && dims_c <= vdim), "head_norm_rotate: a rotation over %d of %d numbers of a value", dims_c, vdim);
    TL_REQUIRE(!k_plane || (v_plane && heads_c == heads_b && heads_c > 0 && positions && token_req && block_table && table_width > 0 && table_ld >= table_width && pages > 0 && page_size > 0),
               "head_norm_rotate: keys and values for the pages need as many heads of each, positions, planes and a block table");
    TL_REQUIRE(!raw_b || raw_ld >= heads_b * dim, "head_norm_rotate: the rows of the copy are too short");
    TL_REQUIRE(tokens >= 0 && heads_a >= 0 && heads_b >= 0 && heads_a + heads_b > 0 && dim > 0 && dim <= LA_MAX_DIM && ld >= (heads_a + heads_b) * dim,
               "head_norm_rotate: bad sizes");
    TL_REQUIRE(!inv_freq || (positions && dims > 0 && dims % 2 == 0 && dims <= dim), "head_norm_rotate: a rotation over %d of %d numbers", dims, dim);
    TL_REQUIRE((norm_a == nullptr) == (norm_b == nullptr) || heads_a == 0 || heads_b == 0, "head_norm_rotate: a norm for both kinds of heads or for neither");
    if (tokens == 0) return TL_OK;
    const long items = (long)tokens * (heads_a + heads_b + heads_c);
    const ValueHeads values{heads_c, vdim, unit_c, (const float*)inv_freq_c, dims_c, halves_c};
    const int grid = (int)((items + HNR_WAVES - 1) / HNR_WAVES);
    if (dtype == TL_DT_F32)
        head_norm_rotate_kernel<float><<<grid, HNR_WAVES * TL_WAVE, 0, stream>>>((float*)x, ld, tokens, heads_a, heads_b, dim, (const float*)norm_a,
            (const float*)norm_b, eps, (const int*)positions, (const float*)inv_freq, dims, halves, (float*)raw_b, raw_ld, magnitude, unit, heat, values,
            PagesOf<float>{(const int*)token_req, (const int*)block_table, table_ld, table_width, (float*)k_plane, (float*)v_plane, pages, page_size});
    else if (dtype == TL_DT_BF16)
        head_norm_rotate_kernel<bf16_t><<<grid, HNR_WAVES * TL_WAVE, 0, stream>>>((bf16_t*)x, ld, tokens, heads_a, heads_b, dim, (const float*)norm_a,
            (const float*)norm_b, eps, (const int*)positions, (const float*)inv_freq, dims, halves, (bf16_t*)raw_b, raw_ld, magnitude, unit, heat, values,
            PagesOf<bf16_t>{(const int*)token_req, (const int*)block_table, table_ld, table_width, (bf16_t*)k_plane, (bf16_t*)v_plane, pages, page_size});
    else TL_REQUIRE(false, "head_norm_rotate: unknown dtype %d", dtype);
    TL_CHECK_LAUNCH("head_norm_rotate");
    return TL_OK;
}
