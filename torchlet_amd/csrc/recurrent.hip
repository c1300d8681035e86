// Recurrent mixers with a fixed-size state per request: the matrix-memory recurrence (mLSTM), the gated delta rule behind its
// short convolutions, a recurrence whose decays are each key channel's and each token's own (the time mixing of RWKV), and the gated per-head norm of their outputs.  State, gates, decays and the output's quotient are float whatever the
// activation type; queries, keys and values come in the activation type as the projection left them.
#include <limits.h>

#include "common.h"
#include <type_traits>

// A barrier that orders shared memory only: __syncthreads() also waits for every fetch from memory that is on its
// way (its fence covers global memory), which would end a prefetch at the first barrier after it.
__device__ __forceinline__ void shared_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// ------------------------------------------------------------------ gates
__device__ __forceinline__ float soft_cap(float z, float cap) { return cap > 0.f ? cap * tanhf(z / cap) : z; }
__device__ __forceinline__ float log_sigmoid(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }

// ------------------------------------------------------------------ the recurrence
// Per request and head a state of dim x vdim numbers S, dim numbers n and a running maximum m:
//   m' = max(f + m, i);  S' = exp(f + m - m') S + exp(i - m') k v^T;  n' likewise with k alone;
//   o  = S'^T q / (max(|n' . q|, exp(-m')) + denom_eps),        q scaled by qscale.
// n is one more column of S, the one whose "value" is 1 for every token: S'[:, n] = keep S[:, n] + take k, and n . q is
// that column's output.  A work-group owns COLS - 1 columns of one request's and head's S and a copy of the n column
// (so nothing is exchanged between work-groups; the first one stores n and m, and all of them read n and m from a
// copy taken before the launch, since a work-group may start after the first one has finished).  A lane owns one column and RPT rows of
// it, in registers for all tokens of the step: with COLS = 64 a wave holds RPT rows, with 32 or 16 it holds two or
// four groups of RPT rows side by side, which makes more and smaller work-groups where a step has few requests.
// Tokens are taken TB at a time: their q, k, v go to shared memory, one wave turns their gates into decays (the capped
// gates and the exponentials side by side, the running maximum one token after the other, as it is defined), every
// lane runs the TB updates of its rows and leaves its rows' shares of each token's sums, and the shares are added in the
// order of the rows.  A share is always that of four rows, whatever RPT and COLS are (a lane with RPT rows leaves RPT / 4
// of them), so a token's result does not depend on the tile's shape: a prompt is run with
// few rows to a lane, because the time of a token is the chain of one lane's updates, a decode step with many rows and
// wide tiles, because its time is the stream of the states.  Long portions leave this loop for the chunks at the end of this file, whose sums are
// in another order: a portion equals single steps to the bit up to the length where that starts, and within rounding beyond it.
#define MLSTM_TB 16
#define MLSTM_SHARE 4

template <typename T, int RPT, int COLS>
__global__ void __launch_bounds__(1024)
mlstm_scan_kernel(const T* __restrict__ qkv, int ld, int k_off, int v_off,
                  const float* __restrict__ gates,          // [tokens, 2 * heads]: raw input gates, raw forget gates
                  float* __restrict__ state, size_t slot_stride, const int* __restrict__ slots, const float* __restrict__ before,
                  const int* __restrict__ req_indptr, float* __restrict__ out, int heads, int dim, int vdim,
                  float cap, float qscale, float denom_eps, int tb, int below) {
    constexpr int RG = TL_WAVE / COLS;                 // groups of RPT rows a wave holds side by side
    extern __shared__ float smem[];
    const int waves = blockDim.x / TL_WAVE, wave = threadIdx.x / TL_WAVE, lane = threadIdx.x % TL_WAVE;
    constexpr int SPL = RPT / MLSTM_SHARE;             // shares of a lane
    const int shares = waves * RG * SPL;               // >= ceil(dim / 4)
    // tb <= MLSTM_TB tokens are taken at a time: no more than the longest request of the step brings, so that a decode step's
    // work-groups need little shared memory and several fit a compute unit
    float* sq = smem;                                  // [tb][dim]
    float* sk = sq + tb * dim;                         // [tb][dim]
    float* sv = sk + tb * dim;                         // [tb][COLS]: the values of the tile's columns, 1 for the n column
    float* sd = sv + tb * COLS;                        // [tb][4]: keep, take, m after the token, (log input gate)
    float* part = sd + tb * 4;                         // [tb][shares][COLS]

    const int req = blockIdx.z, head = blockIdx.y, col0 = blockIdx.x * (COLS - 1);
    const int tok0 = req_indptr[req], tok1 = req_indptr[req + 1];
    if (tok0 >= tok1 || tok1 - tok0 >= below) return;  // (a long portion goes through the chunks)
    const int c = lane % COLS, share = (wave * RG + lane / COLS) * SPL;     // the first of this lane's shares
    const bool is_n = c == COLS - 1;
    const int col = col0 + c;
    const bool col_ok = !is_n && col < vdim;
    const int row0 = share * MLSTM_SHARE;
    float* st = state + (size_t)slots[req] * slot_stride + (size_t)head * ((size_t)dim * vdim + dim + 1);
    float* st_n = st + (size_t)dim * vdim;
    const float* nm = before + ((size_t)req * heads + head) * (dim + 1);      // n and m as they were before the launch

    float S[RPT];
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
        const int row = row0 + r;
        S[r] = row < dim ? (is_n ? nm[row] : (col_ok ? st[(size_t)row * vdim + col] : 0.f)) : 0.f;
    }
    float m = nm[dim];                                 // (kept by the first wave, which turns the gates into decays)

    // A batch's q, k, v and raw gates are fetched into registers while the batch before is worked on (16-byte pieces of the
    // q and k rows where they are aligned), and go to shared memory, widened, when its sums have been read.
    constexpr int VEC = 16 / (int)sizeof(T);           // numbers of a 16-byte piece
    constexpr int QK_PF = (MLSTM_TB * 2 * RPT * RG + VEC * TL_WAVE - 1) / (VEC * TL_WAVE);     // pieces a thread fetches at most
    constexpr int V_PF = MLSTM_TB * COLS / TL_WAVE;    // values a thread fetches at most
    const bool vec_ok = dim % VEC == 0 && ld % VEC == 0 && k_off % VEC == 0 && ((uintptr_t)qkv % 16) == 0;
    const int dv = dim / VEC;
    uint4 qk_stage[QK_PF];
    T v_stage[V_PF];
    float g_stage[2] = {0.f, 0.f};
    auto fetch = [&](int base) {
        const int nb = min(tb, tok1 - base);
        if (vec_ok) {
#pragma unroll
            for (int j = 0; j < QK_PF; ++j) {
                const int idx = min((int)threadIdx.x + j * (int)blockDim.x, nb * 2 * dv - 1);       // (clamped: every lane fetches)
                const int t = idx / (2 * dv), rem = idx % (2 * dv);
                qk_stage[j] = *(const uint4*)(qkv + (size_t)(base + t) * ld + head * dim + (rem >= dv ? k_off : 0) + (rem % dv) * VEC);
            }
        }
#pragma unroll
        for (int j = 0; j < V_PF; ++j) {
            const int idx = min((int)threadIdx.x + j * (int)blockDim.x, nb * COLS - 1);
            const int vc = min(col0 + idx % COLS, vdim - 1);
            v_stage[j] = qkv[(size_t)(base + idx / COLS) * ld + v_off + head * vdim + vc];
        }
        if (wave == 0) {
            const float* g = gates + (size_t)(base + min(lane, nb - 1)) * 2 * heads;
            g_stage[0] = g[head];
            g_stage[1] = g[heads + head];
        }
    };
    fetch(tok0);
    for (int base = tok0; base < tok1; base += tb) {
        const int nb = min(tb, tok1 - base);
        shared_barrier();                               // the sums of the tokens before have been read
        if (vec_ok) {
#pragma unroll
            for (int j = 0; j < QK_PF; ++j) {
                const int idx = threadIdx.x + j * blockDim.x;
                if (idx < nb * 2 * dv) {
                    const int t = idx / (2 * dv), rem = idx % (2 * dv);
                    const bool is_k = rem >= dv;
                    float* dst = (is_k ? sk : sq) + t * dim + (rem % dv) * VEC;
                    const T* piece = (const T*)&qk_stage[j];
#pragma unroll
                    for (int e = 0; e < VEC; ++e) dst[e] = is_k ? to_float(piece[e]) : to_float(piece[e]) * qscale;
                }
            }
        } else {
            for (int i = threadIdx.x; i < nb * dim; i += blockDim.x) {
                const int t = i / dim, d = i % dim;
                const T* row = qkv + (size_t)(base + t) * ld + head * dim;
                sq[t * dim + d] = to_float(row[d]) * qscale;
                sk[t * dim + d] = to_float(row[k_off + d]);
            }
        }
#pragma unroll
        for (int j = 0; j < V_PF; ++j) {
            const int idx = threadIdx.x + j * blockDim.x;
            if (idx < nb * COLS) {
                const int cc = idx % COLS;
                sv[idx] = cc == COLS - 1 ? 1.f : (col0 + cc < vdim ? to_float(v_stage[j]) : 0.f);
            }
        }
        if (wave == 0) {
            // the capped gates side by side, the running maximum token after token (every lane walks the same chain),
            // then the decays side by side
            const float gi = soft_cap(g_stage[0], cap), gf = log_sigmoid(soft_cap(g_stage[1], cap));
            float m_before = m, m_mine = m;
            for (int t = 0; t < nb; ++t) {             // (lane t's gates, read across the wave without a trip to shared memory)
                const float fi = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(gi), t));
                const float ff = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(gf), t));
                const float m_new = fmaxf(ff + m, fi);
                if (lane == t) { m_before = m; m_mine = m_new; }
                m = m_new;
            }
            if (lane < nb) {
                sd[lane * 4] = expf(gf + m_before - m_mine);
                sd[lane * 4 + 1] = expf(gi - m_mine);
                sd[lane * 4 + 2] = m_mine;
            }
        }
        if (base + tb < tok1) fetch(base + tb);
        shared_barrier();
#pragma unroll 4
        for (int t = 0; t < nb; ++t) {
            const float keep = sd[t * 4], tv = sd[t * 4 + 1] * sv[t * COLS + c];
            const float* kt = sk + t * dim + row0;
            const float* qt = sq + t * dim + row0;
#pragma unroll
            for (int u = 0; u < SPL; ++u) {
                float o = 0.f;
#pragma unroll
                for (int r = MLSTM_SHARE * u; r < MLSTM_SHARE * (u + 1); ++r) {
                    if (row0 + r < dim) {
                        S[r] = fmaf(kt[r], tv, keep * S[r]);
                        o = fmaf(S[r], qt[r], o);
                    }
                }
                part[((size_t)t * shares + share + u) * COLS + c] = o;
            }
        }
        shared_barrier();
        for (int t = wave; t < nb; t += waves) {
            if (lane < COLS) {
                // the shares in four interleaved sums (shares 0, 4, 8, ...; 1, 5, 9, ...; ...), added up in their order:
                // one fixed order whatever the work-group's shape, and four chains of additions instead of one
                float o4[4] = {0.f, 0.f, 0.f, 0.f}, n4[4] = {0.f, 0.f, 0.f, 0.f};
                for (int w = 0; w < shares; w += 4) {          // (shares is a multiple of four or the tail is zeros of lanes without rows)
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        if (w + u < shares) {
                            const float* p = part + ((size_t)t * shares + w + u) * COLS;
                            o4[u] += p[lane];
                            n4[u] += p[COLS - 1];
                        }
                    }
                }
                const float osum = ((o4[0] + o4[1]) + o4[2]) + o4[3], nq = ((n4[0] + n4[1]) + n4[2]) + n4[3];
                if (lane < COLS - 1 && col0 + lane < vdim)
                    out[((size_t)(base + t) * heads + head) * vdim + col0 + lane] = osum / (fmaxf(fabsf(nq), expf(-sd[t * 4 + 2])) + denom_eps);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
        const int row = row0 + r;
        if (row < dim) {
            if (col_ok) st[(size_t)row * vdim + col] = S[r];
            else if (is_n && blockIdx.x == 0) st_n[row] = S[r];
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) st_n[dim] = m;
}

// n and m of the step's requests and heads, copied out of their slots: before[(req, head)] = [n (dim), m].
__global__ void mlstm_before_kernel(const float* __restrict__ state, size_t slot_stride, const int* __restrict__ slots,
                                    float* __restrict__ before, int heads, int dim, int vdim) {
    const int req = blockIdx.x / heads, head = blockIdx.x % heads;
    const float* src = state + (size_t)slots[req] * slot_stride + (size_t)head * ((size_t)dim * vdim + dim + 1) + (size_t)dim * vdim;
    float* dst = before + (size_t)blockIdx.x * (dim + 1);
    for (int i = threadIdx.x; i <= dim; i += blockDim.x) dst[i] = src[i];
}

template <typename T, int RPT, int COLS>
static int launch_mlstm_scan(const void* qkv, int ld, int k_off, int v_off, const void* gates, void* state, size_t slot_stride,
                             const void* slots, const void* before, const void* req_indptr, void* out, int requests, int heads, int dim, int vdim,
                             float cap, float qscale, float denom_eps, int tb, int below, hipStream_t stream) {
    constexpr int RG = TL_WAVE / COLS;
    const int waves = (dim + RPT * RG - 1) / (RPT * RG);
    TL_REQUIRE(waves <= 16, "mlstm_scan: %d rows of a head do not fit a work-group of %d rows a lane and %d columns", dim, RPT, COLS);
    // tokens of a batch: as many as asked for, halved until their inputs and sums fit the shared memory (large heads)
    const size_t per_token = sizeof(float) * ((size_t)2 * dim + COLS + 4 + (size_t)waves * RG * (RPT / MLSTM_SHARE) * COLS);
    while (tb > 1 && per_token * tb > 144 * 1024) tb /= 2;
    const size_t smem = per_token * tb;
    TL_REQUIRE(smem <= 160 * 1024, "mlstm_scan: %zu bytes of shared memory for dim %d", smem, dim);
    auto kernel = mlstm_scan_kernel<T, RPT, COLS>;
    static size_t allowed = 48 * 1024;               // (per instance of the template)
    if (smem > allowed) {
        hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
        if (e != hipSuccess) { tl_set_error("mlstm_scan: cannot get %zu bytes of shared memory: %s", smem, hipGetErrorString(e)); return TL_ERR_HIP; }
        allowed = smem;
    }
    dim3 grid((vdim + COLS - 2) / (COLS - 1), heads, requests), block(waves * TL_WAVE);
    mlstm_before_kernel<<<requests * heads, 128, 0, stream>>>((const float*)state, slot_stride, (const int*)slots, (float*)before, heads, dim, vdim);
    TL_CHECK_LAUNCH("mlstm_before");
    kernel<<<grid, block, smem, stream>>>((const T*)qkv, ld, k_off, v_off, (const float*)gates, (float*)state, slot_stride,
                                           (const int*)slots, (const float*)before, (const int*)req_indptr, (float*)out, heads, dim, vdim, cap, qscale, denom_eps, tb, below);
    TL_CHECK_LAUNCH("mlstm_scan");
    return TL_OK;
}

static int tl_mlstm_units = 256;       // compute units the column tiles are dealt to
extern "C" void tl_mlstm_set_compute_units(int units) { if (units > 0) tl_mlstm_units = units; }

// Columns of a work-group: as few as it takes to give every compute unit one (the sums do not depend on the choice); rows a lane keeps: as few as 16 waves
// of such lanes can hold the head's rows with, four at least.
struct MlstmShape { int cols, rpt; };
static MlstmShape mlstm_shape(int requests, int heads, int dim, int vdim) {
    const long heads_reqs = (long)heads * requests;
    const int cols = heads_reqs * ((vdim + 62) / 63) >= tl_mlstm_units ? 64 : heads_reqs * ((vdim + 30) / 31) >= tl_mlstm_units ? 32 : 16;
    const int need = (dim * cols + 16 * TL_WAVE - 1) / (16 * TL_WAVE);
    return {cols, need <= 4 ? 4 : need <= 8 ? 8 : need <= 16 ? 16 : need <= 32 ? 32 : 64};
}

// The token loop: requests of `below` tokens or more are left alone.
static int mlstm_token_loop(const void* qkv, int ld, int k_off, int v_off, const void* gates, void* state, long slot_stride,
                            const void* slots, const void* before, const void* req_indptr, void* out, int requests, int heads, int dim, int vdim,
                            float cap, float qscale, float denom_eps, int longest, int below, int dtype, hipStream_t stream) {
    TL_REQUIRE(requests >= 0 && heads > 0 && dim > 0 && vdim > 0 && ld > 0, "mlstm_scan: bad sizes");
    const int tb = longest < 1 ? 1 : (longest < MLSTM_TB ? longest : MLSTM_TB);       // longest: the most tokens a request of the step brings
    TL_REQUIRE(dim <= 1024, "mlstm_scan: built for up to 1024 query/key dimensions per head, got %d", dim);
    TL_REQUIRE(slot_stride >= (long)heads * ((long)dim * vdim + dim + 1), "mlstm_scan: the state rows are too short");
    TL_REQUIRE(dtype == TL_DT_F32 || dtype == TL_DT_BF16, "mlstm_scan: unknown dtype %d", dtype);
    if (requests == 0) return TL_OK;
    const MlstmShape shape = mlstm_shape(requests, heads, dim, vdim);
    const int cols = shape.cols, rpt = shape.rpt;
#define TL_MLSTM_C(R, C)                                                                                                       \
    return dtype == TL_DT_F32                                                                                                  \
        ? launch_mlstm_scan<float, R, C>(qkv, ld, k_off, v_off, gates, state, (size_t)slot_stride, slots, before, req_indptr, out,    \
                                         requests, heads, dim, vdim, cap, qscale, denom_eps, tb, below, stream)                      \
        : launch_mlstm_scan<bf16_t, R, C>(qkv, ld, k_off, v_off, gates, state, (size_t)slot_stride, slots, before, req_indptr, out,   \
                                          requests, heads, dim, vdim, cap, qscale, denom_eps, tb, below, stream)
#define TL_MLSTM(R)                                  \
    if (cols == 64) { TL_MLSTM_C(R, 64); }           \
    else if (cols == 32) { TL_MLSTM_C(R, 32); }      \
    else { TL_MLSTM_C(R, 16); }
    switch (rpt) {
        case 4: TL_MLSTM(4)
        case 8: TL_MLSTM(8)
        case 16: TL_MLSTM(16)
        case 32: TL_MLSTM(32)
        default: TL_MLSTM(64)
    }
#undef TL_MLSTM
#undef TL_MLSTM_C
}

// ------------------------------------------------------------------ gated per-head norm
// y[t, h, :] = o[t, h, :] / sqrt(mean(o[t, h, :]^2) + eps) * weight[h, :] * gate(g[t, h, :]) * gain; one wave per token and head.
// gate 0: sigmoid, 1: silu.  shared_weight: one vector of vdim numbers for all heads.  The rows of g and y may be longer than
// heads * vdim (views into wider buffers).  gate_first: the gate comes before the norm, y = u / sqrt(mean(u^2) + eps) * weight * gain
// with u = o * gate(g) (a "head" is then whatever stretch of the row is normed together).
template <typename T>
__global__ void gated_head_norm_kernel(const float* __restrict__ o, const T* __restrict__ gate, int gate_ld,
                                       const void* __restrict__ weight, int weight_f32, int shared_weight, float eps,
                                       T* __restrict__ out, int out_ld, int rows, int heads, int vdim, int gate_kind, float gain, int gate_first) {
    const int row = blockIdx.x * (blockDim.x / TL_WAVE) + threadIdx.x / TL_WAVE, lane = threadIdx.x % TL_WAVE;
    if (row >= rows) return;
    const int t = row / heads, h = row % heads;
    const float* src = o + (size_t)row * vdim;
    const T* g = gate + (size_t)t * gate_ld + h * vdim;
    float ss = 0.f;
    for (int i = lane; i < vdim; i += TL_WAVE) {
        float u = src[i];
        if (gate_first) {
            const float z = to_float(g[i]);
            const float s = 1.f / (1.f + expf(-z));
            u *= gate_kind == 1 ? z * s : s;
        }
        ss = fmaf(u, u, ss);
    }
    ss = wave_sum(ss);
    const float inv = 1.f / sqrtf(ss / (float)vdim + eps);
    T* dst = out + (size_t)t * out_ld + h * vdim;
    const int w0 = shared_weight ? 0 : h * vdim;
    for (int i = lane; i < vdim; i += TL_WAVE) {
        const float z = to_float(g[i]);
        const float s = 1.f / (1.f + expf(-z));
        dst[i] = from_float<T>(src[i] * (gate_kind == 1 ? z * s : s) * inv * load_vec(weight, weight_f32, w0 + i) * gain);
    }
}

// The same for long stretches (more than 512 numbers normed together: all heads of a mixer as one): a work-group of 256 threads per token and
// stretch instead of a wave, the sum of squares joined through shared memory.
template <typename T>
__global__ void __launch_bounds__(256)
gated_row_norm_kernel(const float* __restrict__ o, const T* __restrict__ gate, int gate_ld, const void* __restrict__ weight, int weight_f32,
                      int shared_weight, float eps, T* __restrict__ out, int out_ld, int heads, int vdim, int gate_kind, float gain, int gate_first) {
    __shared__ float red[16];
    const int row = blockIdx.x;
    const int t = row / heads, h = row % heads;
    const float* src = o + (size_t)row * vdim;
    const T* g = gate + (size_t)t * gate_ld + h * vdim;
    float ss = 0.f;
    for (int i = threadIdx.x; i < vdim; i += blockDim.x) {
        float u = src[i];
        if (gate_first) {
            const float z = to_float(g[i]);
            const float s = 1.f / (1.f + expf(-z));
            u *= gate_kind == 1 ? z * s : s;
        }
        ss = fmaf(u, u, ss);
    }
    ss = block_sum(ss, red);
    const float inv = 1.f / sqrtf(ss / (float)vdim + eps);
    T* dst = out + (size_t)t * out_ld + h * vdim;
    const int w0 = shared_weight ? 0 : h * vdim;
    for (int i = threadIdx.x; i < vdim; i += blockDim.x) {
        const float z = to_float(g[i]);
        const float s = 1.f / (1.f + expf(-z));
        dst[i] = from_float<T>(src[i] * (gate_kind == 1 ? z * s : s) * inv * load_vec(weight, weight_f32, w0 + i) * gain);
    }
}

// The same with a stretch's numbers in registers: LANES threads to a stretch (part of a wave, a wave, or a work-group of its own), NP pieces of four
// neighbouring numbers to a thread, all requested before the first is used, so that a stretch costs one trip to memory instead of one per number
// of a thread and pass.  What bounds it is its bytes on prompts and its launch and that one trip in decode steps: 4 tokens of 4096 numbers 15.3 -> 4.0 us, of
// 8192 27.5 -> 5.4 us (one number a thread and trip before). 
template <typename T, int NP, int LANES>
__global__ void __launch_bounds__(LANES > 256 ? LANES : 256)
gated_norm_pieces_kernel(const float* __restrict__ o, const T* __restrict__ gate, int gate_ld, const void* __restrict__ weight, int weight_f32,
                         int shared_weight, float eps, T* __restrict__ out, int out_ld, int rows, int heads, int vdim, int gate_kind, float gain, int gate_first) {
    __shared__ float red[16];
    const int row = LANES > 256 ? blockIdx.x : blockIdx.x * (256 / LANES) + threadIdx.x / LANES, lane = threadIdx.x % LANES;
    const bool live = row < rows;                       // (rows beyond the last one take part in the exchanges)
    const int t = live ? row / heads : 0, h = live ? row % heads : 0;
    const float* src = o + ((size_t)t * heads + h) * vdim;
    const T* g = gate + (size_t)t * gate_ld + (size_t)h * vdim;
    const size_t w0 = shared_weight ? 0 : (size_t)h * vdim;
    float4 u[NP], f[NP], wv[NP];
    typename Four<T>::type raw[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const int at = (lane + p * LANES) * 4;
        if (at < vdim) {
            u[p] = *(const float4*)(src + at);
            raw[p] = *(const typename Four<T>::type*)(g + at);
            wv[p] = weight_f32 ? *(const float4*)((const float*)weight + w0 + at) : widen4(*(const ushort4*)((const bf16_t*)weight + w0 + at));
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        if ((lane + p * LANES) * 4 < vdim) {
            const float4 z = widen4(raw[p]);
            const float4 s = make_float4(1.f / (1.f + expf(-z.x)), 1.f / (1.f + expf(-z.y)), 1.f / (1.f + expf(-z.z)), 1.f / (1.f + expf(-z.w)));
            f[p] = gate_kind == 1 ? make_float4(z.x * s.x, z.y * s.y, z.z * s.z, z.w * s.w) : s;
            const float4 v = gate_first ? make_float4(u[p].x * f[p].x, u[p].y * f[p].y, u[p].z * f[p].z, u[p].w * f[p].w) : u[p];
            ss = fmaf(v.x, v.x, ss); ss = fmaf(v.y, v.y, ss); ss = fmaf(v.z, v.z, ss); ss = fmaf(v.w, v.w, ss);
        }
    }
    if constexpr (LANES > TL_WAVE) ss = block_sum(ss, red);
    else ss = lanes_sum<LANES>(ss);
    const float inv = 1.f / sqrtf(ss / (float)vdim + eps);
    if (!live) return;
    T* dst = out + (size_t)t * out_ld + (size_t)h * vdim;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const int at = (lane + p * LANES) * 4;
        if (at < vdim)
            store4(dst + at, make_float4(u[p].x * f[p].x * inv * wv[p].x * gain, u[p].y * f[p].y * inv * wv[p].y * gain,
                                         u[p].z * f[p].z * inv * wv[p].z * gain, u[p].w * f[p].w * inv * wv[p].w * gain));
    }
}

// Pieces of four where every row and vector lets a lane read them whole, and stretches of up to 16384 numbers; number by number otherwise.
template <typename T>
static bool gated_norm_pieces(const void* o, const void* gate, int gate_ld, const void* weight, int weight_f32, int shared_weight, float eps, void* out,
                              int out_ld, int rows, int heads, int vdim, int gate_kind, float gain, int gate_first, hipStream_t stream) {
    constexpr size_t piece = 4 * sizeof(T);
    if (vdim % 4 || gate_ld % 4 || out_ld % 4 || vdim > 16384 || ((uintptr_t)o | (uintptr_t)weight) % 16
        || ((uintptr_t)gate | (uintptr_t)out) % piece) return false;
#define TL_GN(NP, LANES)                                                                                                                          \
    gated_norm_pieces_kernel<T, NP, LANES><<<LANES > 256 ? rows : (rows + 256 / LANES - 1) / (256 / LANES), LANES > 256 ? LANES : 256, 0, stream>>>( \
        (const float*)o, (const T*)gate, gate_ld, weight, weight_f32, shared_weight, eps, (T*)out, out_ld, rows, heads, vdim, gate_kind, gain, gate_first)
    if (vdim <= 64) TL_GN(1, 16);
    else if (vdim <= 128) TL_GN(1, 32);
    else if (vdim <= 256) TL_GN(1, 64);
    else if (vdim <= 512) TL_GN(2, 64);
    else if (vdim <= 2048) TL_GN(1, 512);
    else if (vdim <= 4096) TL_GN(1, 1024);
    else if (vdim <= 8192) TL_GN(2, 1024);
    else TL_GN(4, 1024);
#undef TL_GN
    return true;
}

extern "C" int tl_gated_head_norm(const void* o, const void* gate, int gate_ld, const void* weight, int weight_f32, int shared_weight, float eps,
                                  void* out, int out_ld, int tokens, int heads, int vdim, int gate_kind, float gain, int gate_first, int dtype,
                                  hipStream_t stream) {
    TL_REQUIRE(tokens >= 0 && heads > 0 && vdim > 0 && gate_ld >= heads * vdim && out_ld >= heads * vdim, "gated_head_norm: bad sizes");
    TL_REQUIRE(gate_kind == 0 || gate_kind == 1, "gated_head_norm: unknown gate %d", gate_kind);
    if (tokens == 0) return TL_OK;
    const int rows = tokens * heads;
    TL_REQUIRE(dtype == TL_DT_F32 || dtype == TL_DT_BF16, "gated_head_norm: unknown dtype %d", dtype);
    if (dtype == TL_DT_F32 ? gated_norm_pieces<float>(o, gate, gate_ld, weight, weight_f32, shared_weight, eps, out, out_ld, rows, heads, vdim, gate_kind, gain, gate_first, stream)
                           : gated_norm_pieces<bf16_t>(o, gate, gate_ld, weight, weight_f32, shared_weight, eps, out, out_ld, rows, heads, vdim, gate_kind, gain, gate_first, stream)) {
        TL_CHECK_LAUNCH("gated_norm_pieces");
        return TL_OK;
    }
    if (vdim > 512) {
        if (dtype == TL_DT_F32)
            gated_row_norm_kernel<float><<<rows, 256, 0, stream>>>((const float*)o, (const float*)gate, gate_ld, weight, weight_f32, shared_weight, eps,
                                                                   (float*)out, out_ld, heads, vdim, gate_kind, gain, gate_first);
        else if (dtype == TL_DT_BF16)
            gated_row_norm_kernel<bf16_t><<<rows, 256, 0, stream>>>((const float*)o, (const bf16_t*)gate, gate_ld, weight, weight_f32, shared_weight, eps,
                                                                    (bf16_t*)out, out_ld, heads, vdim, gate_kind, gain, gate_first);
        else TL_REQUIRE(false, "gated_head_norm: unknown dtype %d", dtype);
        TL_CHECK_LAUNCH("gated_row_norm");
        return TL_OK;
    }
    dim3 grid((rows + 3) / 4), block(4 * TL_WAVE);
    if (dtype == TL_DT_F32)
        gated_head_norm_kernel<float><<<grid, block, 0, stream>>>((const float*)o, (const float*)gate, gate_ld, weight, weight_f32, shared_weight, eps,
                                                                  (float*)out, out_ld, rows, heads, vdim, gate_kind, gain, gate_first);
    else if (dtype == TL_DT_BF16)
        gated_head_norm_kernel<bf16_t><<<grid, block, 0, stream>>>((const float*)o, (const bf16_t*)gate, gate_ld, weight, weight_f32, shared_weight, eps,
                                                                   (bf16_t*)out, out_ld, rows, heads, vdim, gate_kind, gain, gate_first);
    else TL_REQUIRE(false, "gated_head_norm: unknown dtype %d", dtype);
    TL_CHECK_LAUNCH("gated_head_norm");
    return TL_OK;
}

// ------------------------------------------------------------------ gated delta rule: what the recurrence reads
// A token's convolved channels come in units: kv_heads query heads, kv_heads key heads (dim channels each), heads value heads (vdim
// channels each); one wave per token and unit.  Channel c at the request's i-th token of the step:
//   y = sum_j w[c][j] * x[i - (taps - 1) + j][c],   x[i'] = the projection of the step's token i' >= 0, else tail[taps - 1 + i'][c]
//   (the slot's last taps - 1 inputs from before the step, oldest first; zero for a new request), then silu;
//   query and key heads: y / sqrt(sum y^2 + unit_eps), queries times qscale.
// One more unit per token turns the raw gates into beta = sigmoid(b) and decay = exp(-exp(a_log) * softplus(a + dt_bias)).
#define DELTA_MAX_TAPS 8
#define DELTA_UNIT_MAX 4        // channels a lane holds: heads of up to 256 channels

__device__ __forceinline__ float silu_f(float z) { return z / (1.f + expf(-z)); }
__device__ __forceinline__ float softplus_f(float z) { return z > 20.f ? z : log1pf(expf(z)); }

template <typename T>
__global__ void __launch_bounds__(256)
delta_prepare_kernel(const T* __restrict__ proj, int ld, const float* __restrict__ conv_w, float* __restrict__ gates,
                     const float* __restrict__ a_log, const float* __restrict__ dt_bias, const float* __restrict__ state, size_t slot_stride,
                     size_t tail_off, const int* __restrict__ slots, const int* __restrict__ req_indptr, const int* __restrict__ token_req,
                     float* __restrict__ qkv, int heads, int kv_heads, int dim, int vdim, int taps, float qscale, float unit_eps) {
    const int t = blockIdx.x, lane = threadIdx.x % TL_WAVE;
    const int unit = blockIdx.y * (blockDim.x / TL_WAVE) + threadIdx.x / TL_WAVE;
    const int units = 2 * kv_heads + heads;
    if (unit > units) return;
    if (unit == units) {                               // the gates of the token's heads
        for (int h = lane; h < heads; h += TL_WAVE) {
            float* g = gates + (size_t)t * 2 * heads;
            const float b = g[h], a = g[heads + h];
            g[h] = 1.f / (1.f + expf(-b));
            g[heads + h] = expf(-expf(a_log[h]) * softplus_f(a + dt_bias[h]));
        }
        return;
    }
    const int C = 2 * kv_heads * dim + heads * vdim;
    const bool is_v = unit >= 2 * kv_heads;
    const int width = is_v ? vdim : dim;
    const int c0 = is_v ? 2 * kv_heads * dim + (unit - 2 * kv_heads) * vdim : unit * dim;
    const int req = token_req[t];
    const int i = t - req_indptr[req];                 // the token's place in its request's portion
    const float* tail = state + (size_t)slots[req] * slot_stride + tail_off;
    float y[DELTA_UNIT_MAX];
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < DELTA_UNIT_MAX; ++u) {
        const int c = c0 + lane + u * TL_WAVE;
        y[u] = 0.f;
        if (lane + u * TL_WAVE < width) {
            float acc = 0.f;
            for (int j = 0; j < taps; ++j) {
                const int back = i - (taps - 1) + j;   // the input's place in the portion
                const float xv = back >= 0 ? to_float(proj[(size_t)(t - i + back) * ld + c]) : tail[(size_t)(taps - 1 + back) * C + c];
                acc = fmaf(conv_w[(size_t)c * taps + j], xv, acc);
            }
            y[u] = silu_f(acc);
            ss = fmaf(y[u], y[u], ss);
        }
    }
    float factor = 1.f;
    if (!is_v) {
        ss = wave_sum(ss);
        factor = 1.f / sqrtf(ss + unit_eps);
        if (unit < kv_heads) factor *= qscale;
    }
#pragma unroll
    for (int u = 0; u < DELTA_UNIT_MAX; ++u)
        if (lane + u * TL_WAVE < width) qkv[(size_t)t * C + c0 + lane + u * TL_WAVE] = y[u] * factor;
}

// After the step the tail of a request holds the last taps - 1 inputs of its channels: of the step's tokens, and before those of the
// old tail.  A thread owns a channel of a request and reads the old tail before it writes.
template <typename T>
__global__ void delta_tail_kernel(const T* __restrict__ proj, int ld, float* __restrict__ state, size_t slot_stride, size_t tail_off,
                                  const int* __restrict__ slots, const int* __restrict__ req_indptr, int C, int taps) {
    const int req = blockIdx.y, c = blockIdx.x * blockDim.x + threadIdx.x;
    const int tok0 = req_indptr[req], n = req_indptr[req + 1] - tok0;
    if (c >= C || n <= 0) return;
    float* tail = state + (size_t)slots[req] * slot_stride + tail_off;
    float old[DELTA_MAX_TAPS];
#pragma unroll
    for (int j = 0; j < DELTA_MAX_TAPS - 1; ++j) old[j] = j < taps - 1 ? tail[(size_t)j * C + c] : 0.f;
#pragma unroll
    for (int j = 0; j < DELTA_MAX_TAPS - 1; ++j) {
        if (j < taps - 1) {
            const int back = n - (taps - 1) + j;       // place in the portion of what becomes entry j
            float v = 0.f;
            if (back >= 0) v = to_float(proj[(size_t)(tok0 + back) * ld + c]);
            else {
#pragma unroll
                for (int q = 0; q < DELTA_MAX_TAPS - 1; ++q)
                    if (q == j + n) v = old[q];
            }
            tail[(size_t)j * C + c] = v;
        }
    }
}

// ------------------------------------------------------------------ short convolutions in pieces
// What delta_prepare_kernel and selective_prepare_kernel (MODE 1) make, for four taps and channels that come in whole pieces of four: a thread owns four
// neighbouring channels of a run of RUN tokens (their taps, and the window of the three inputs before the current token, stay in registers), so an input is
// fetched once instead of once per tap, 8 or 16 bytes at a time, and the run's inputs are requested together.  A head's unit norm is shared by the dim / 4
// neighbouring lanes that hold it.  OWN: for steps with as many tokens as requests (decode steps), without the tail's launch: a work-group takes the first three tokens of the
// request of its own number, the only ones that read its tail, moves the tail on (its threads own the channels they read), and takes the token of its own number if that
// is a later one of its request: whatever a request brings, nobody walks its tokens one after the other (one request of 2048 tokens of 4096 channels beside 2047 empty ones
// 1830 us when the request's work-group did, 18.7 now; 16 requests of one token 3.4 both ways).
// Bound by its bytes on prompts (2048 tokens of 4096 channels 53 -> 20 us, 3000 of 8448 163 -> 43 us), by launch and one trip to memory in decode steps (with the tail's kernel
// 11.3 -> 4.5 us).
struct ConvArgs {
    const float *w, *bias;           // [C][4]; [C] or null
    float* gates;
    const float *a_log, *dt_bias;
    float* state;
    size_t slot_stride, tail_off;
    const int *slots, *req_indptr, *token_req;
    float* out;
    int ld, C, tokens, heads;
    int q_end, unit_end, unit_lanes;         // MODE 0: channels of queries, of queries and keys; lanes of a head
    float qscale, unit_eps;
    int inner, gn;                           // MODE 1
};

template <typename T, int RUN, int MODE, bool OWN>
__global__ void __launch_bounds__(256)
short_conv_kernel(const T* __restrict__ proj, ConvArgs a) {
    const int p = blockIdx.y * 256 + threadIdx.x, pieces = a.C / 4, gate0 = (pieces + TL_WAVE - 1) / TL_WAVE * TL_WAVE;
    const int first = OWN ? a.req_indptr[blockIdx.x] : (int)blockIdx.x * RUN;
    const int end = OWN ? a.req_indptr[blockIdx.x + 1] : min(first + RUN, a.tokens), last = OWN ? min(first + 3, end) : end;
    const bool more = OWN && (int)blockIdx.x - a.req_indptr[a.token_req[blockIdx.x]] >= 3;
    if (p >= gate0) {                                  // (whole waves) the gates of the tokens' heads
        const int h = p - gate0;
        if (h >= a.heads) return;
        for (int t = OWN ? (int)blockIdx.x : first; t < (OWN ? (int)blockIdx.x + 1 : last); ++t) {
            float* g = a.gates + (size_t)t * 2 * a.heads;
            if (MODE == 0) {
                const float b = g[h], v = g[a.heads + h];
                g[h] = 1.f / (1.f + expf(-b));
                g[a.heads + h] = expf(-expf(a.a_log[h]) * softplus_f(v + a.dt_bias[h]));
            } else {
                const float dt = softplus_f(to_float(proj[(size_t)t * a.ld + a.C + h]) + a.dt_bias[h]);
                g[h] = dt;
                g[a.heads + h] = expf(-expf(a.a_log[h]) * dt);
            }
        }
        return;
    }
    typedef typename Four<T>::type Piece;
    const bool live = p < pieces;
    const int c = live ? 4 * p : 0;
    const T* col = proj + c;
    float4 tap[4];                                     // tap[e]: the four taps of channel c + e
#pragma unroll
    for (int e = 0; e < 4; ++e) tap[e] = *(const float4*)(a.w + (size_t)(c + e) * 4);
    const float4 bias = MODE == 1 ? *(const float4*)(a.bias + c) : make_float4(0.f, 0.f, 0.f, 0.f);
    float4 win[3];
    int req = -1;
    float* tail = nullptr;
    auto convolve = [&](int t, const float4& now) {
        float4 y = bias;
#define TL_TAP(f, e) y.f = fmaf(tap[e].w, now.f, fmaf(tap[e].z, win[2].f, fmaf(tap[e].y, win[1].f, fmaf(tap[e].x, win[0].f, y.f))))
        TL_TAP(x, 0); TL_TAP(y, 1); TL_TAP(z, 2); TL_TAP(w, 3);
#undef TL_TAP
        y = make_float4(silu_f(y.x), silu_f(y.y), silu_f(y.z), silu_f(y.w));
        int to = c;
        if (MODE == 0) {
            float ss = fmaf(y.w, y.w, fmaf(y.z, y.z, fmaf(y.y, y.y, y.x * y.x)));
            for (int k = a.unit_lanes / 2; k > 0; k >>= 1) ss += __shfl_xor(ss, k, TL_WAVE);
            if (c < a.unit_end) {
                float factor = 1.f / sqrtf(ss + a.unit_eps);
                if (c < a.q_end) factor *= a.qscale;
                y = make_float4(y.x * factor, y.y * factor, y.z * factor, y.w * factor);
            }
        } else {
            to = c < a.inner ? 2 * a.gn + c : (c < a.inner + a.gn ? a.gn + (c - a.inner) : c - a.inner - a.gn);
        }
        if (live) store4(a.out + (size_t)t * a.C + to, y);
    };
    for (int base = first; base < last; base += RUN) {
        Piece x[RUN];
#pragma unroll
        for (int u = 0; u < RUN; ++u) x[u] = *(const Piece*)(col + (size_t)min(base + u, last - 1) * a.ld);
#pragma unroll
        for (int u = 0; u < RUN; ++u) {
            const int t = base + u;
            if (t >= last) break;
            const int r = OWN ? (int)blockIdx.x : a.token_req[t];
            if (r != req) {                            // the window before the run's, or a request's, first token
                req = r;
                const int tok0 = a.req_indptr[r], i = t - tok0;
                tail = a.state + (size_t)a.slots[r] * a.slot_stride + a.tail_off + c;
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    const int back = i - 3 + j;
                    if (back >= 0) win[j] = widen4(*(const Piece*)(col + (size_t)(tok0 + back) * a.ld));
                    else win[j] = *(const float4*)(tail + (size_t)(3 + back) * a.C);
                }
            }
            const float4 now = widen4(x[u]);
            convolve(t, now);
            win[0] = win[1]; win[1] = win[2]; win[2] = now;
        }
    }
    if (OWN && live && end > first) {
#pragma unroll
        for (int j = 0; j < 3; ++j) store4(tail + (size_t)j * a.C, end - first > 3 ? widen4(*(const Piece*)(col + (size_t)(end - 3 + j) * a.ld)) : win[j]);
    }
    if (more) {                                        // (a wave together)
        const int t = blockIdx.x;
#pragma unroll
        for (int j = 0; j < 3; ++j) win[j] = widen4(*(const Piece*)(col + (size_t)(t - 3 + j) * a.ld));
        convolve(t, widen4(*(const Piece*)(col + (size_t)t * a.ld)));
    }
}

// Whether the pieces fit (four taps, aligned rows; a head's lanes a power of two inside a wave); then the launch: OWN for steps of as many tokens as requests,
// else the tail's launch is the caller's.  Runs of eight tokens where that leaves every compute unit several work-groups, of two below.
template <typename T, int MODE>
static bool short_conv(const T* proj, ConvArgs a, int requests, hipStream_t stream, bool* tail_done) {
    const uintptr_t bits = (uintptr_t)a.w | (uintptr_t)a.bias | (uintptr_t)a.state | (uintptr_t)a.out;
    if (bits % 16 || (uintptr_t)proj % (4 * sizeof(T)) || a.ld % 4 || a.C % 4 || a.slot_stride % 4 || a.tail_off % 4) return false;
    if (MODE == 0 && (a.unit_lanes > TL_WAVE || (a.unit_lanes & (a.unit_lanes - 1)) || a.unit_end % 4)) return false;
    if (MODE == 1 && (a.inner % 4 || a.gn % 4)) return false;
    const int gate0 = (a.C / 4 + TL_WAVE - 1) / TL_WAVE * TL_WAVE, blocks = (gate0 + a.heads + 255) / 256;
    if (blocks > 65535) return false;
    *tail_done = a.tokens == requests;
    if (a.tokens == requests) short_conv_kernel<T, 1, MODE, true><<<dim3(requests, blocks), 256, 0, stream>>>(proj, a);
    else if ((long)a.tokens * blocks >= 8 * 1024) short_conv_kernel<T, 8, MODE, false><<<dim3((a.tokens + 7) / 8, blocks), 256, 0, stream>>>(proj, a);
    else short_conv_kernel<T, 2, MODE, false><<<dim3((a.tokens + 1) / 2, blocks), 256, 0, stream>>>(proj, a);
    return true;
}

extern "C" int tl_delta_prepare(const void* proj, int ld, const void* conv_w, void* gates, const void* a_log, const void* dt_bias, void* state,
                                long slot_stride, long tail_off, const void* slots, const void* req_indptr, const void* token_req, void* qkv,
                                int tokens, int requests, int heads, int kv_heads, int dim, int vdim, int taps, float qscale, float unit_eps,
                                int dtype, hipStream_t stream) {
    TL_REQUIRE(tokens >= 0 && requests >= 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && vdim > 0, "delta_prepare: bad sizes");
    TL_REQUIRE(taps >= 1 && taps <= DELTA_MAX_TAPS, "delta_prepare: 1 to %d taps are built, not %d", DELTA_MAX_TAPS, taps);
    TL_REQUIRE(dim <= DELTA_UNIT_MAX * TL_WAVE && vdim <= DELTA_UNIT_MAX * TL_WAVE, "delta_prepare: heads of up to %d channels are built", DELTA_UNIT_MAX * TL_WAVE);
    const int C = 2 * kv_heads * dim + heads * vdim;
    TL_REQUIRE(ld >= C && tail_off >= 0 && slot_stride >= tail_off + (long)(taps - 1) * C, "delta_prepare: rows or state too short");
    TL_REQUIRE(dtype == TL_DT_F32 || dtype == TL_DT_BF16, "delta_prepare: unknown dtype %d", dtype);
    if (tokens == 0 || requests == 0) return TL_OK;
    const int units = 2 * kv_heads + heads + 1;
    dim3 grid(tokens, (units + 3) / 4), block(4 * TL_WAVE);
    dim3 tgrid((C + 255) / 256, requests), tblock(256);
    if (taps == 4 && dim % 4 == 0 && vdim % 4 == 0) {
        ConvArgs a = {(const float*)conv_w, nullptr, (float*)gates, (const float*)a_log, (const float*)dt_bias, (float*)state, (size_t)slot_stride, (size_t)tail_off,
                      (const int*)slots, (const int*)req_indptr, (const int*)token_req, (float*)qkv, ld, C, tokens, heads,
                      kv_heads * dim, 2 * kv_heads * dim, dim / 4, qscale, unit_eps, 0, 0};
        bool tail_done = false;
        if (dtype == TL_DT_F32 ? short_conv<float, 0>((const float*)proj, a, requests, stream, &tail_done)
                               : short_conv<bf16_t, 0>((const bf16_t*)proj, a, requests, stream, &tail_done)) {
            TL_CHECK_LAUNCH("delta_prepare");
            if (tail_done) return TL_OK;
            if (dtype == TL_DT_F32) delta_tail_kernel<float><<<tgrid, tblock, 0, stream>>>((const float*)proj, ld, (float*)state, (size_t)slot_stride, (size_t)tail_off,
                                                                                           (const int*)slots, (const int*)req_indptr, C, taps);
            else delta_tail_kernel<bf16_t><<<tgrid, tblock, 0, stream>>>((const bf16_t*)proj, ld, (float*)state, (size_t)slot_stride, (size_t)tail_off,
                                                                         (const int*)slots, (const int*)req_indptr, C, taps);
            TL_CHECK_LAUNCH("delta_tail");
            return TL_OK;
        }
    }
    if (dtype == TL_DT_F32) {
        delta_prepare_kernel<float><<<grid, block, 0, stream>>>((const float*)proj, ld, (const float*)conv_w, (float*)gates, (const float*)a_log, (const float*)dt_bias,
            (const float*)state, (size_t)slot_stride, (size_t)tail_off, (const int*)slots, (const int*)req_indptr, (const int*)token_req, (float*)qkv,
            heads, kv_heads, dim, vdim, taps, qscale, unit_eps);
        TL_CHECK_LAUNCH("delta_prepare");
        if (taps > 1) delta_tail_kernel<float><<<tgrid, tblock, 0, stream>>>((const float*)proj, ld, (float*)state, (size_t)slot_stride, (size_t)tail_off,
                                                                             (const int*)slots, (const int*)req_indptr, C, taps);
    } else {
        delta_prepare_kernel<bf16_t><<<grid, block, 0, stream>>>((const bf16_t*)proj, ld, (const float*)conv_w, (float*)gates, (const float*)a_log, (const float*)dt_bias,
            (const float*)state, (size_t)slot_stride, (size_t)tail_off, (const int*)slots, (const int*)req_indptr, (const int*)token_req, (float*)qkv,
            heads, kv_heads, dim, vdim, taps, qscale, unit_eps);
        TL_CHECK_LAUNCH("delta_prepare");
        if (taps > 1) delta_tail_kernel<bf16_t><<<tgrid, tblock, 0, stream>>>((const bf16_t*)proj, ld, (float*)state, (size_t)slot_stride, (size_t)tail_off,
                                                                              (const int*)slots, (const int*)req_indptr, C, taps);
    }
    TL_CHECK_LAUNCH("delta_tail");
    return TL_OK;
}

// ------------------------------------------------------------------ gated delta rule: the recurrence
// Per request and head a state S of dim x vdim numbers; per token, with the decay g, the step size beta, unit q (scaled) and k:
//   S <- g S;   u = beta (v - S^T k);   S <- S + k u^T;   o = S^T q.
// Column j of S needs only its own a_j = sum_r S[r][j] k[r] and b_j = sum_r S[r][j] q[r] (of the state before the decay) and k . q:
//   u_j = beta (v_j - g a_j);   o_j = g b_j + (k . q) u_j;   S[r][j] <- g S[r][j] + k[r] u_j.
// The 16 lanes of a row of the wave share a column: lane i of them owns the rows 64 q + 4 i .. + 3 (q < RPL / 4; RPL = 4, 8, 12 or 16, fixed
// by dim alone) of it in registers for all tokens of the step, so the lanes' pieces of q and k lie side by side in shared memory and those of
// the state side by side in memory ([vdim][dim] per head), and they add their sums with four exchanges inside the row (pairs, quads, halves,
// the row: every lane gets the same bits).  k . q, which all columns share, is made once a token.  The order of every sum is fixed by dim, so a
// token's result in this loop depends neither on how its request was cut into steps nor on what else the step holds.  (Long portions leave it, fixed decays for chunks of 64 tokens and the other
// two for blocks of 16, see below, where a step's sizes make that the faster way: from CHUNKED_FROM or BLOCKS_FROM tokens on a portion's rounding depends on where it was cut and, through
// that choice, on what else the step holds.)  A wave has 4 CPL columns, a work-group
// of four waves 16 CPL.  Tokens are taken TB at a time (1, 4 or 16, by the longest portion of the step): their q, k, v, beta and g are fetched
// into registers one batch ahead, as whole pieces of four where the rows allow it, and go to shared memory; a request's last batch is filled up
// with tokens that change nothing (k = 0, beta = 0, decay 1), so the loop has no branch.
// What bounds it: a token is a chain (S -> a -> u -> S) of some 50 vector instructions a wave beside six reads of shared memory; the fetches and
// their address arithmetic must stay small beside that (number by number, each under a condition of its own, they were five sixths of the
// instructions and held a work-group at 256 registers).  Measured: see launch_delta_scan.
#define DELTA_L 16
#define DELTA_COLS 16           // columns of a work-group
#define DELTA_TB 16

template <int CTRL>
__device__ __forceinline__ float row_exchange(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}

// The sum of v over the 16 lanes of a row of the wave, in every one of them.
__device__ __forceinline__ float row16_sum(float v) {
    v += row_exchange<0xB1>(v);        // quad_perm [1, 0, 3, 2]: the neighbour
    v += row_exchange<0x4E>(v);        // quad_perm [2, 3, 0, 1]: the other pair of the quad
    v += row_exchange<0x141>(v);       // row_half_mirror: the other quad of the half
    v += row_exchange<0x140>(v);       // row_mirror: the other half
    return v;
}

// MODE 1: the delta rule.  MODE 0: the same recurrence without the correction, S <- g S + k v^T and o = S^T q, with one fixed decay per
// head (`head_decay`) in place of the tokens' gates: the decayed linear attention.  MODE 2: without the correction, with the tokens' own
// decays and step sizes, S <- g S + k (beta v)^T and o = S^T q + skip v with one skip factor per head (`head_decay` holds them): a
// selective state-space recurrence (k: the input matrix's row B, q: the output matrix's row C, beta: the step size, v: the input).
template <int RPL, int TB, int MODE, int CPL>
__global__ void __launch_bounds__(256, RPL * CPL <= 16 ? 4 : 2)
delta_scan_kernel(const float* __restrict__ qkv, const float* __restrict__ gates, const float* __restrict__ head_decay,
                  float* __restrict__ state, size_t slot_stride,
                  const int* __restrict__ slots, const int* __restrict__ req_indptr, float* __restrict__ out,
                  int heads, int kv_heads, int dim, int vdim, int vec, int below) {
    constexpr int ROWS = DELTA_L * RPL, Q = RPL / 4, COLS = DELTA_COLS * CPL;          // ROWS >= dim
    constexpr int PPT = ROWS / 4, NP = (TB * PPT + 255) / 256, NV = (TB * COLS + 255) / 256;      // pieces of four: per token, per thread and batch
    __shared__ __attribute__((aligned(16))) float sq[TB * ROWS], sk[TB * ROWS], sg[TB * 4];       // sg: beta, decay, k . q
    __shared__ float sv[TB * COLS];
    const int req = blockIdx.z, head = blockIdx.y, col0 = blockIdx.x * COLS;
    const int tok0 = req_indptr[req], tok1 = req_indptr[req + 1];
    if (tok0 >= tok1 || tok1 - tok0 >= below) return;            // (a long portion goes through the chunks)
    const int tid = threadIdx.x, wave = tid / TL_WAVE, lane = tid % TL_WAVE;
    const int rg = lane & 15, cw = wave * 4 + (lane >> 4);       // the lane's place in its columns, and the first of them within the work-group
    const int C = 2 * kv_heads * dim + heads * vdim;
    const int qk_head = head / (heads / kv_heads);
    const int q_at = qk_head * dim, k_at = kv_heads * dim + qk_head * dim, v_at = 2 * kv_heads * dim + head * vdim + col0;
    float* st = state + (size_t)slots[req] * slot_stride + (size_t)head * vdim * dim;

    float S[CPL][RPL];
    const bool vec_state = (dim & 3) == 0 && ((uintptr_t)state & 15) == 0 && (slot_stride & 3) == 0;
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        const int col = col0 + cw + c * DELTA_COLS;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int row = 64 * q + 4 * rg;
            const float* from = st + (size_t)col * dim + row;
            if (vec_state && col < vdim && row + 4 <= dim) {
                const float4 x = *(const float4*)from;
                S[c][4 * q] = x.x; S[c][4 * q + 1] = x.y; S[c][4 * q + 2] = x.z; S[c][4 * q + 3] = x.w;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) S[c][4 * q + e] = (col < vdim && row + e < dim) ? from[e] : 0.f;
            }
        }
    }

    // The state is waited for here: left to the token loop, the wait at its head would be one for every fetch on its way, the next batch's too.
#pragma unroll
    for (int c = 0; c < CPL; ++c)
#pragma unroll
        for (int r = 0; r < RPL; ++r) asm volatile("" : "+v"(S[c][r]));

    float4 pq[NP], pk[NP];
    float pv[NV], pg = 0.f;
    auto fetch = [&](int base) {
        const int nb = min(TB, tok1 - base);
        if (vec && nb == TB && (TB * PPT) % 256 == 0) {           // whole pieces of whole tokens, and one for every thread
#pragma unroll
            for (int j = 0; j < NP; ++j) {
                const int idx = tid + j * 256;
                const float* row = qkv + (size_t)(base + idx / PPT) * C + (idx % PPT) * 4;
                pq[j] = *(const float4*)(row + q_at);
                pk[j] = *(const float4*)(row + k_at);
            }
        } else if (vec) {
#pragma unroll
            for (int j = 0; j < NP; ++j) {
                const int idx = tid + j * 256, t = idx / PPT;
                const float* row = qkv + (size_t)(base + t) * C + (idx % PPT) * 4;
                pq[j] = pk[j] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (idx < TB * PPT && t < nb) {
                    pq[j] = *(const float4*)(row + q_at);
                    pk[j] = *(const float4*)(row + k_at);
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < NP; ++j) {
                const int idx = tid + j * 256, t = idx / PPT, e = (idx % PPT) * 4;
                pq[j] = pk[j] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (idx < TB * PPT && t < nb && e < dim) {
                    const float* row = qkv + (size_t)(base + t) * C + e;
                    float a[4], b[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        a[u] = e + u < dim ? row[q_at + u] : 0.f;
                        b[u] = e + u < dim ? row[k_at + u] : 0.f;
                    }
                    pq[j] = make_float4(a[0], a[1], a[2], a[3]);
                    pk[j] = make_float4(b[0], b[1], b[2], b[3]);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int idx = tid + j * 256, t = idx / COLS, c = idx % COLS;
            pv[j] = (idx < TB * COLS && t < nb && col0 + c < vdim) ? qkv[(size_t)(base + t) * C + v_at + c] : 0.f;
        }
        if (tid < 2 * TB) {                            // beyond the request's last token: k = 0, beta = 0 and a decay of 1 leave the state as it is, to the bit
            const int t = tid >> 1, which = tid & 1;
            if (t >= nb) pg = which ? 1.f : 0.f;
            else if (MODE != 0) pg = gates[(size_t)(base + t) * 2 * heads + which * heads + head];
            else pg = which ? head_decay[head] : 1.f;
        }
    };
    const float skip = MODE == 2 ? head_decay[head] : 0.f;
    fetch(tok0);
    for (int base = tok0; base < tok1; base += TB) {
        const int nb = min(TB, tok1 - base);
        shared_barrier();                              // the batch before has been worked on
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const int idx = tid + j * 256;
            if (idx < TB * PPT) {
                *(float4*)(sq + idx * 4) = pq[j];
                *(float4*)(sk + idx * 4) = pk[j];
            }
        }
#pragma unroll
        for (int j = 0; j < NV; ++j)
            if (tid + j * 256 < TB * COLS) sv[tid + j * 256] = pv[j];
        if (tid < 2 * TB) sg[(tid >> 1) * 4 + (tid & 1)] = pg;
        if (base + TB < tok1) fetch(base + TB);
        shared_barrier();
        // k . q: the 16 lanes of column cw make token cw's
        if (cw < TB) {
            float c4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const float4 k4 = *(const float4*)(sk + cw * ROWS + 64 * q + 4 * rg), q4 = *(const float4*)(sq + cw * ROWS + 64 * q + 4 * rg);
                c4[0] = fmaf(k4.x, q4.x, c4[0]);
                c4[1] = fmaf(k4.y, q4.y, c4[1]);
                c4[2] = fmaf(k4.z, q4.z, c4[2]);
                c4[3] = fmaf(k4.w, q4.w, c4[3]);
            }
            const float kq = row16_sum((c4[0] + c4[1]) + (c4[2] + c4[3]));
            if (rg == 0) sg[cw * 4 + 2] = kq;
        }
        shared_barrier();
        float mine[CPL];                               // the outputs of token rg of the batch
#pragma unroll
        for (int c = 0; c < CPL; ++c) mine[c] = 0.f;
        // a token's operands are read from shared memory one token ahead, beside the sums of the token at hand (asked for when they are needed,
        // four tokens' at a time, they and the sums took turns)
        float4 kn[Q], qn[Q], gn;
        float vn[CPL];
        auto ahead = [&](int t) {
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                kn[q] = *(const float4*)(sk + t * ROWS + 64 * q + 4 * rg);
                qn[q] = *(const float4*)(sq + t * ROWS + 64 * q + 4 * rg);
            }
            gn = *(const float4*)(sg + t * 4);
#pragma unroll
            for (int c = 0; c < CPL; ++c) vn[c] = sv[t * COLS + cw + c * DELTA_COLS];
        };
        ahead(0);
#pragma unroll 4
        for (int t = 0; t < TB; ++t) {
            float kr[RPL], qr[RPL], vr[CPL];
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                kr[4 * q] = kn[q].x; kr[4 * q + 1] = kn[q].y; kr[4 * q + 2] = kn[q].z; kr[4 * q + 3] = kn[q].w;
                qr[4 * q] = qn[q].x; qr[4 * q + 1] = qn[q].y; qr[4 * q + 2] = qn[q].z; qr[4 * q + 3] = qn[q].w;
            }
#pragma unroll
            for (int c = 0; c < CPL; ++c) vr[c] = vn[c];
            const float beta = gn.x, g = gn.y, kq = gn.z;
            ahead(min(t + 1, TB - 1));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                const float vt = vr[c];
                // four chains of additions each, joined in a fixed order
                float a4[4] = {0.f, 0.f, 0.f, 0.f}, b4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int r = 0; r < RPL; ++r) {
                    if (MODE == 1) a4[r & 3] = fmaf(S[c][r], kr[r], a4[r & 3]);
                    b4[r & 3] = fmaf(S[c][r], qr[r], b4[r & 3]);
                }
                const float a = MODE == 1 ? row16_sum((a4[0] + a4[1]) + (a4[2] + a4[3])) : 0.f;
                const float b = row16_sum((b4[0] + b4[1]) + (b4[2] + b4[3]));
                const float u = MODE == 1 ? beta * fmaf(-g, a, vt) : (MODE == 2 ? beta * vt : vt);
#pragma unroll
                for (int r = 0; r < RPL; ++r) S[c][r] = fmaf(kr[r], u, g * S[c][r]);
                const float o = MODE == 2 ? fmaf(skip, vt, fmaf(kq, u, g * b)) : fmaf(kq, u, g * b);
                if (rg == t) mine[c] = o;
            }
        }
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            const int col = col0 + cw + c * DELTA_COLS;
            if (rg < nb && col < vdim) out[((size_t)(base + rg) * heads + head) * vdim + col] = mine[c];
        }
    }
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        const int col = col0 + cw + c * DELTA_COLS;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int row = 64 * q + 4 * rg;
            float* to = st + (size_t)col * dim + row;
            if (vec_state && col < vdim && row + 4 <= dim) *(float4*)to = make_float4(S[c][4 * q], S[c][4 * q + 1], S[c][4 * q + 2], S[c][4 * q + 3]);
            else if (col < vdim) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (row + e < dim) to[e] = S[c][4 * q + e];
            }
        }
    }
}

// Columns of a lane: two (half the reads of shared memory a column) where one to a lane would not all be on the GPU at once, four work-groups to a
// compute unit; up to there more waves win.  What counts as on the GPU at once is the step's work over that of its longest request (a request's last batch is
// worked through whole): beside a long prompt the work-groups of decoded requests are gone after one batch.  Measured (us, one column / two; number-by-number
// fetches before): the delta rule, 16 heads of 128 x 128, one prompt of 2048 tokens 405 / 603 (1533), beside 8 decoded tokens 418 / 605, eight prompts of 175 to 700
// tokens 189 / 230 (1328); the selective recurrence, 128 heads of 128 x 64, four prompts of 275 to 1100 tokens 467 / 342 (3780); fixed decays, 16 heads of
// 128 x 128, 2048 tokens 366 / 492 (1342).  Portions of 4 tokens and single ones (8 requests, 9 us) as before.
static int delta_columns(int dim, int vdim, int heads, int requests, int tokens, int longest) {
    if (dim > 128 || longest <= 4) return 1;
    const double longs = ((double)tokens + (DELTA_TB - 1.0) * requests) / (longest < DELTA_TB ? DELTA_TB : longest);
    return (double)((vdim + DELTA_COLS - 1) / DELTA_COLS) * heads * longs > 4.0 * tl_mlstm_units ? 2 : 1;
}
// (the rule alone, for tests)
extern "C" int tl_delta_columns(int dim, int vdim, int heads, int requests, int tokens, int longest) { return delta_columns(dim, vdim, heads, requests, tokens, longest); }

// state: per slot, from its start, heads x [vdim][dim] floats (a head's state column by column).
template <int MODE>
static int launch_delta_scan(const void* qkv, const void* gates, const void* head_decay, void* state, long slot_stride, const void* slots,
                             const void* req_indptr, void* out, int requests, int heads, int kv_heads, int dim, int vdim, int tokens, int longest, int below, hipStream_t stream) {
    const int rpl = dim <= 64 ? 4 : dim <= 128 ? 8 : dim <= 192 ? 12 : 16;
    // tokens of a batch: 1 for a step of single tokens, 4 for short portions, else 16 (a batch is always worked through whole)
    const int tb = longest <= 1 ? 1 : (longest <= 4 ? 4 : DELTA_TB);
    const int vec = dim == DELTA_L * rpl && vdim % 4 == 0 && ((uintptr_t)qkv & 15) == 0;       // (a token's numbers are then a multiple of four)
    const int cpl = delta_columns(dim, vdim, heads, requests, tokens, longest);
    dim3 grid((vdim + DELTA_COLS * cpl - 1) / (DELTA_COLS * cpl), heads, requests), block(256);
#define TL_DELTA_B(R, B, P)                                                                                                                \
    delta_scan_kernel<R, B, MODE, P><<<grid, block, 0, stream>>>((const float*)qkv, (const float*)gates, (const float*)head_decay, (float*)state, \
                                                           (size_t)slot_stride, (const int*)slots, (const int*)req_indptr, (float*)out, heads, kv_heads, dim, vdim, vec, below)
#define TL_DELTA(R)                           \
    if (tb == 1) TL_DELTA_B(R, 1, 1);         \
    else if (tb == 4) TL_DELTA_B(R, 4, 1);    \
    else TL_DELTA_B(R, DELTA_TB, 1)
    if (cpl == 2 && rpl == 4) TL_DELTA_B(4, DELTA_TB, 2);
    else if (cpl == 2 && rpl == 8) TL_DELTA_B(8, DELTA_TB, 2);
    else if (rpl == 4) { TL_DELTA(4); }
    else if (rpl == 8) { TL_DELTA(8); }
    else if (rpl == 12) { TL_DELTA(12); }
    else { TL_DELTA(16); }
#undef TL_DELTA
#undef TL_DELTA_B
    return TL_OK;
}

// ------------------------------------------------------------------ the delta rule's single tokens: convolution, recurrence, norm and gate in one launch
// For steps of one token a request: what short_conv_kernel (four taps), delta_scan_kernel and gated_norm_pieces_kernel (silu, one weight for all heads) make in three launches, in the same
// order of every sum.  A work-group has a key head of a request with the value heads that share it, so the channels it convolves, and the tail it moves on, are its own.  It asks for
// its states first, sixteen lanes a column and CG columns to each; while they are on their way the convolution's inputs arrive, its threads make q, k, v and the heads' gates and leave them in
// shared memory, then all lanes move the states, and the first ones take the outputs through the norm.  What bounds it: a compute unit draws the states of its work-group at 64 bytes a clock, 128 KB
// for two value heads of 128 x 128, and gives them back as fast.  8 requests, 16 heads of 128 x 128 over 8: 4.5 + 6.8 + 4.1 us in three launches, 9.3 in one; calls one behind the other, gaps included, 1
// request 7.9 and 6.6 us, 8 10.7 and 7.6, 32 20.6 and 12.2, 64 32.2 and 27.2, 128 52.5 and 50.6 (198 registers leave a unit one work-group; it is ahead at every size measured, up to 3072 of them).
// Built for key heads of 64 or 128 channels with up to 256 value channels between them.
#define DT_THREADS 512                          // (sixteen waves leave a wave 128 registers, which 256 columns of 128 do not fit)
#define DT_COLS (DT_THREADS / DELTA_L)           // columns at a time
struct DeltaToken {
    int ld, gate_off;
    const float *w, *gates, *a_log, *dt_bias;
    float* state;
    size_t slot_stride, tail_off;
    const int *slots, *req_indptr;
    const float* norm;
    float eps, gain, qscale, unit_eps;
    int out_ld, heads, kv_heads, vdim;
};
template <typename T, int RPL, int CG>
__global__ void __launch_bounds__(DT_THREADS)
delta_token_kernel(const T* __restrict__ proj, T* __restrict__ out, DeltaToken a) {
    constexpr int dim = DELTA_L * RPL, Q = RPL / 4, U = dim / 4;         // U: lanes of a key head's channels
    __shared__ __attribute__((aligned(16))) float sq[dim], sk[dim], sv[CG * DT_COLS], so[CG * DT_COLS], sg[2 * CG * DT_COLS];
    const int req = blockIdx.y, kv = blockIdx.x;
    const int slot_at = a.slots[req], tok0 = a.req_indptr[req], tok1 = a.req_indptr[req + 1];
    if (tok0 >= tok1) return;
    const int tid = threadIdx.x, rg = tid & 15, cw = tid >> 4, vdim = a.vdim, hpk = a.heads / a.kv_heads, cols = hpk * vdim, head0 = kv * hpk;
    const int C = 2 * a.kv_heads * dim + a.heads * vdim;
    float* slot = a.state + (size_t)slot_at * a.slot_stride;
    float* st = slot + (size_t)head0 * vdim * dim;                  // the value heads' columns, one behind the other
    float4 S[CG][Q];
#pragma unroll
    for (int c = 0; c < CG; ++c)
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int col = c * DT_COLS + cw;
            S[c][q] = *(const float4*)(st + (size_t)min(col, cols - 1) * dim + 64 * q + 4 * rg);
        }
    // the convolution's threads: four neighbouring channels each, queries, keys, then values
    const int pieces = 2 * U + cols / 4;
    const bool conv = tid < pieces;
    const int p = min(tid, pieces - 1);
    const int ch = p < U ? kv * dim + 4 * p : p < 2 * U ? (a.kv_heads + kv) * dim + 4 * (p - U) : 2 * a.kv_heads * dim + head0 * vdim + 4 * (p - 2 * U);
    float* tail = slot + a.tail_off + ch;
    const bool conv_wave = tid < (pieces + TL_WAVE - 1) / TL_WAVE * TL_WAVE;      // (its last lanes make the last piece again and store nothing)
    float4 tap[4], win[3];
    if (conv_wave) {
#pragma unroll
        for (int j = 0; j < 3; ++j) win[j] = *(const float4*)(tail + (size_t)j * C);
#pragma unroll
        for (int e = 0; e < 4; ++e) tap[e] = *(const float4*)(a.w + (size_t)(ch + e) * 4);
    }
    // the norm's threads: LANES lanes to a value head
    const int lanes = vdim <= 64 ? 16 : 32, hn = tid / lanes, n_at = tid % lanes * 4;
    const bool norms = hn < hpk, n_ok = norms && n_at < vdim;
    for (int t = tok0; t < tok1; ++t) {
        const T* row = proj + (size_t)t * a.ld;
        typename Four<T>::type gate{};
        float4 nw = make_float4(0.f, 0.f, 0.f, 0.f);
        if (n_ok) {
            gate = *(const typename Four<T>::type*)(row + a.gate_off + (head0 + hn) * vdim + n_at);
            nw = *(const float4*)(a.norm + n_at);
        }
        if (tid >= DT_THREADS - hpk) {                              // (the last threads have nothing to convolve: there are at most 128 pieces, and 16 heads)
            const int h = DT_THREADS - 1 - tid;
            const float* g = a.gates + (size_t)t * 2 * a.heads + head0 + h;
            sg[2 * h] = 1.f / (1.f + expf(-g[0]));
            sg[2 * h + 1] = expf(-expf(a.a_log[head0 + h]) * softplus_f(g[a.heads] + a.dt_bias[head0 + h]));
        }
        if (conv_wave) {
            const float4 now = load4(row + ch);
            float4 y;
#define TL_TAP(f, e) y.f = silu_f(fmaf(tap[e].w, now.f, fmaf(tap[e].z, win[2].f, fmaf(tap[e].y, win[1].f, fmaf(tap[e].x, win[0].f, 0.f)))))
            TL_TAP(x, 0); TL_TAP(y, 1); TL_TAP(z, 2); TL_TAP(w, 3);
#undef TL_TAP
            const float ss = lanes_sum<U>(fmaf(y.w, y.w, fmaf(y.z, y.z, fmaf(y.y, y.y, y.x * y.x))));
            if (p < 2 * U) {
                float factor = 1.f / sqrtf(ss + a.unit_eps);
                if (p < U) factor *= a.qscale;
                y = make_float4(y.x * factor, y.y * factor, y.z * factor, y.w * factor);
            }
            if (conv) *(float4*)(p < U ? sq + 4 * p : p < 2 * U ? sk + 4 * (p - U) : sv + 4 * (p - 2 * U)) = y;
            win[0] = win[1]; win[1] = win[2]; win[2] = now;
        }
        __syncthreads();
        float4 k4[Q], q4[Q];
        float c4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            k4[q] = *(const float4*)(sk + 64 * q + 4 * rg);
            q4[q] = *(const float4*)(sq + 64 * q + 4 * rg);
            c4[0] = fmaf(k4[q].x, q4[q].x, c4[0]);
            c4[1] = fmaf(k4[q].y, q4[q].y, c4[1]);
            c4[2] = fmaf(k4[q].z, q4[q].z, c4[2]);
            c4[3] = fmaf(k4[q].w, q4[q].w, c4[3]);
        }
        const float kq = row16_sum((c4[0] + c4[1]) + (c4[2] + c4[3]));
#pragma unroll
        for (int c = 0; c < CG; ++c) {
            const int col = c * DT_COLS + cw;
            if (col >= cols) break;                                 // (16 lanes together)
            const int h = col / vdim;
            const float vt = sv[col], beta = sg[2 * h], g = sg[2 * h + 1];
            float a4[4] = {0.f, 0.f, 0.f, 0.f}, b4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const float4 x = S[c][q];
                a4[0] = fmaf(x.x, k4[q].x, a4[0]); a4[1] = fmaf(x.y, k4[q].y, a4[1]); a4[2] = fmaf(x.z, k4[q].z, a4[2]); a4[3] = fmaf(x.w, k4[q].w, a4[3]);
                b4[0] = fmaf(x.x, q4[q].x, b4[0]); b4[1] = fmaf(x.y, q4[q].y, b4[1]); b4[2] = fmaf(x.z, q4[q].z, b4[2]); b4[3] = fmaf(x.w, q4[q].w, b4[3]);
            }
            const float dot = row16_sum((a4[0] + a4[1]) + (a4[2] + a4[3])), b = row16_sum((b4[0] + b4[1]) + (b4[2] + b4[3]));
            const float u = beta * fmaf(-g, dot, vt);
#pragma unroll
            for (int q = 0; q < Q; ++q)
                S[c][q] = make_float4(fmaf(k4[q].x, u, g * S[c][q].x), fmaf(k4[q].y, u, g * S[c][q].y), fmaf(k4[q].z, u, g * S[c][q].z), fmaf(k4[q].w, u, g * S[c][q].w));
            if (rg == 0) so[col] = fmaf(kq, u, g * b);
        }
        __syncthreads();
        if (tid < (hpk * lanes + TL_WAVE - 1) / TL_WAVE * TL_WAVE) {
            const float4 u = n_ok ? *(const float4*)(so + hn * vdim + n_at) : make_float4(0.f, 0.f, 0.f, 0.f), z = widen4(gate);
            float ss = fmaf(u.x, u.x, 0.f);
            ss = fmaf(u.y, u.y, ss); ss = fmaf(u.z, u.z, ss); ss = fmaf(u.w, u.w, ss);
            ss = vdim <= 64 ? lanes_sum<16>(ss) : lanes_sum<32>(ss);
            const float inv = 1.f / sqrtf(ss / (float)vdim + a.eps);
            const float4 f = make_float4(z.x * (1.f / (1.f + expf(-z.x))), z.y * (1.f / (1.f + expf(-z.y))), z.z * (1.f / (1.f + expf(-z.z))), z.w * (1.f / (1.f + expf(-z.w))));
            if (n_ok) store4(out + (size_t)t * a.out_ld + (head0 + hn) * vdim + n_at, make_float4(u.x * f.x * inv * nw.x * a.gain, u.y * f.y * inv * nw.y * a.gain,
                                                                                                  u.z * f.z * inv * nw.z * a.gain, u.w * f.w * inv * nw.w * a.gain));
        }
        // (a request that brings more: the next token's q, k, v and gates go where these were read before the second barrier, its outputs where the norm's waves read behind it)
        if (t + 1 < tok1) __syncthreads();
    }
#pragma unroll
    for (int c = 0; c < CG; ++c) {
        const int col = c * DT_COLS + cw;
#pragma unroll
        for (int q = 0; q < Q; ++q)
            if (col < cols) *(float4*)(st + (size_t)col * dim + 64 * q + 4 * rg) = S[c][q];
    }
    if (conv) {
#pragma unroll
        for (int j = 0; j < 3; ++j) *(float4*)(tail + (size_t)j * C) = win[j];
    }
}

// Whether delta_token_kernel is built for these sizes and places.
extern "C" int tl_delta_token_fits(const void* proj, int ld, int gate_off, const void* conv_w, const void* state, long slot_stride, long tail_off, const void* norm, const void* out, int out_ld,
                                   int heads, int kv_heads, int dim, int vdim, int taps, int dtype) {
    const size_t piece = dtype == TL_DT_F32 ? 16 : 8;
    return (dtype == TL_DT_F32 || dtype == TL_DT_BF16) && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && (dim == 64 || dim == 128) && vdim >= 16 && vdim % 4 == 0 && vdim <= 128 &&
           heads / kv_heads * vdim <= 256 && taps == 4 && (ld | gate_off | out_ld) % 4 == 0 && slot_stride % 4 == 0 && tail_off % 4 == 0 &&
           ((uintptr_t)proj | (uintptr_t)out) % piece == 0 && ((uintptr_t)conv_w | (uintptr_t)state | (uintptr_t)norm) % 16 == 0;
}

// Operands as tl_delta_prepare, tl_delta_scan and tl_gated_head_norm take them; gates stays as it is; the output gate's numbers lie in the rows of proj from gate_off on; norm float [vdim].
extern "C" int tl_delta_token(const void* proj, int ld, int gate_off, const void* conv_w, const void* gates, const void* a_log, const void* dt_bias, void* state, long slot_stride, long tail_off,
                              const void* slots, const void* req_indptr, const void* norm, float eps, float gain, void* out, int out_ld, int requests, int heads, int kv_heads, int dim,
                              int vdim, int taps, float qscale, float unit_eps, int dtype, hipStream_t stream) {
    TL_REQUIRE(requests >= 0 && requests <= 65535 && gates && a_log && dt_bias, "delta_token: bad sizes");
    TL_REQUIRE(tl_delta_token_fits(proj, ld, gate_off, conv_w, state, slot_stride, tail_off, norm, out, out_ld, heads, kv_heads, dim, vdim, taps, dtype),
               "delta_token: not built for %d heads of %d x %d over %d or for these places", heads, dim, vdim, kv_heads);
    const int C = 2 * kv_heads * dim + heads * vdim, cols = heads / kv_heads * vdim;
    TL_REQUIRE(ld >= C && gate_off >= C && ld >= gate_off + heads * vdim && out_ld >= heads * vdim && tail_off >= (long)heads * dim * vdim && slot_stride >= tail_off + 3L * C,
               "delta_token: rows or state too short");
    if (requests == 0) return TL_OK;
    const DeltaToken a{ld, gate_off, (const float*)conv_w, (const float*)gates, (const float*)a_log, (const float*)dt_bias, (float*)state, (size_t)slot_stride, (size_t)tail_off,
                       (const int*)slots, (const int*)req_indptr, (const float*)norm, eps, gain, qscale, unit_eps, out_ld, heads, kv_heads, vdim};
#define TL_DTK(T, R, G) delta_token_kernel<T, R, G><<<dim3(kv_heads, requests), DT_THREADS, 0, stream>>>((const T*)proj, (T*)out, a)
#define TL_DTK_R(T, R) if (cols <= 2 * DT_COLS) TL_DTK(T, R, 2); else if (cols <= 4 * DT_COLS) TL_DTK(T, R, 4); else TL_DTK(T, R, 8)
#define TL_DTK_T(T) if (dim == 64) { TL_DTK_R(T, 4); } else { TL_DTK_R(T, 8); }
    if (dtype == TL_DT_F32) { TL_DTK_T(float); } else { TL_DTK_T(bf16_t); }
#undef TL_DTK_T
#undef TL_DTK_R
#undef TL_DTK
    TL_CHECK_LAUNCH("delta_token");
    return TL_OK;
}

// ------------------------------------------------------------------ long portions in blocks: the delta rule and the selective recurrence
// The token loop above is a chain of some 500 cycles a token, whatever else the GPU does (one prompt of 2048 tokens, 16 heads: 412 us on 128 work-groups).  Over a block of
// 16 tokens the recurrence is a few products of small matrices (the compact form of a product of Householder-like steps, Bischof and Van Loan's WY representation, as "Parallelizing Linear
// Transformers with the Delta Rule over Sequence Length", Yang et al. 2024, use it), with S the state before the block, g the decays, G_i = prod_{l <= i} g_l and D_ij = prod_{j < l <= i} g_l:
//   L_ij = beta_i (k_i . k_j) D_ij below the diagonal;   U = (1 + L)^-1 diag(beta) (V - diag(G) K S);   O = diag(G) Q S + (Q K^T o D) U;   S <- G_16 S + K^T diag(w) U,  w_j = D_16,j
// (the selective recurrence: U = diag(beta) V).  What does not need the state, T = (1 + L)^-1 diag(beta), P = Q K^T o D, G and w, is made for all blocks at once by
// block_matrices_kernel (the inverse by substitution, and the decays' products, in 64 bits; no quotients, so a decay of zero is one); block_scan_kernel then walks a request's
// blocks with the state in registers: products in true 32-bit on v_mfma_f32_16x16x4_f32, whose result layout (lane l: rows 4 (l / 16) + v of column l % 16) is the
// layout of its right operand, so state, U and V never change lanes.  A work-group owns 16 columns, each of four waves a quarter of their rows: one barrier a block, for the
// quarters' shares of K S and Q S; a fifth wave makes the outputs, a block behind.  What bounds it: a block's chain of products (28 matrix instructions of 32 cycles a wave at 128 x 128, four of them one after the other for U), the exchange and a wait for operands, some 2700 cycles for
// 16 tokens: 2048 tokens, 16 heads of 128 x 128 413 -> 162 us.  Errors against 64 bits (1500 tokens, whole outputs; loop / blocks): slow decays 1.5e-7 to 1.75e-7 / 1.0e-7, fast ones 7.0e-8 / 6.5e-8, selective 1.1e-7 / 0.8e-7.
// Requests of few tokens in the step stay with the token loop, whose bits do not depend on how a request is cut into steps; blocks are counted from the step's first token of the request.
#define BL_T 16                 // tokens of a block

typedef float bl_f32x4 __attribute__((ext_vector_type(4)));

// A block's and head's numbers in scratch.
template <int MODE> struct BlockPlaces {
    static constexpr int P = 0, G = 256, W = 272, PD = 288, TD = 304, T = 320, FLOATS = MODE == 1 ? 576 : 304;      // (PD, TD: the diagonals, zero in P and T)
};

__device__ __forceinline__ int bl_blocks(const int* __restrict__ req_indptr, int r, int least) {
    const int n = req_indptr[r + 1] - req_indptr[r];
    return n >= least ? (n + BL_T - 1) / BL_T : 0;
}

// One wave for a block, the heads that share its keys four at a time.
template <int MODE>
__global__ void __launch_bounds__(64)
block_matrices_kernel(const float* __restrict__ qkv, const float* __restrict__ gates, const int* __restrict__ req_indptr, float* __restrict__ scratch,
                      int requests, int heads, int kv_heads, int dim, int vdim, int least) {
    __shared__ double skk[BL_T][BL_T + 1], sqk[BL_T][BL_T + 1], sl[4][BL_T][BL_T + 1];
    __shared__ float sg[4][BL_T], sb[4][BL_T];
    const int lane = threadIdx.x, quad = lane >> 4, c = lane & 15;
    int first = 0, req = -1, block0 = 0;
    for (int base = 0; base < requests && req < 0; base += TL_WAVE) {
        const int r = base + lane;
        const int mine = r < requests ? bl_blocks(req_indptr, r, least) : 0;
        int upto = mine;
#pragma unroll
        for (int o = 1; o < TL_WAVE; o <<= 1) {
            const int t = __shfl_up(upto, o, TL_WAVE);
            if (lane >= o) upto += t;
        }
        const unsigned long long past = __ballot(first + upto > (int)blockIdx.x);
        if (past) {
            const int l = __builtin_amdgcn_readfirstlane(__ffsll(past) - 1);
            req = base + l;
            block0 = first + __builtin_amdgcn_readlane(upto, l) - __builtin_amdgcn_readlane(mine, l);
        }
        first += __builtin_amdgcn_readlane(upto, TL_WAVE - 1);
    }
    if (req < 0) return;                                   // (the grid is an upper bound)
    const int tok0 = req_indptr[req] + ((int)blockIdx.x - block0) * BL_T, nt = min(BL_T, req_indptr[req + 1] - tok0);
    const int C = 2 * kv_heads * dim + heads * vdim, share = heads / kv_heads;
    const int parts = (share + 3) / 4, kv = blockIdx.y / parts, in_share = (blockIdx.y % parts) * 4 + quad;
    const bool live = in_share < share;
    const int head = kv * share + min(in_share, share - 1);
    const float* row = qkv + (size_t)(tok0 + min(c, nt - 1)) * C + kv * dim + 4 * quad;
    // (sums of eight products each, joined in 64 bits: 128 of them in one chain double the error of what the block's own tokens contribute)
    double kk[4] = {0.0, 0.0, 0.0, 0.0}, qk[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 2
    for (int d0 = 0; d0 < dim; d0 += 32) {
        bl_f32x4 ks[4], qs[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) ks[v] = qs[v] = bl_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int d = d0; d < d0 + 32; d += 16) {
            float4 q = make_float4(0.f, 0.f, 0.f, 0.f), k = q;
            if (d + 4 * quad < dim) {
                q = *(const float4*)(row + d);
                k = *(const float4*)(row + kv_heads * dim + d);
            }
            const float qa[4] = {q.x, q.y, q.z, q.w}, ka[4] = {k.x, k.y, k.z, k.w};
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if (MODE == 1) ks[v] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[v], ka[v], ks[v], 0, 0, 0);
                qs[v] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[v], ka[v], qs[v], 0, 0, 0);
            }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            if (MODE == 1) kk[v] += ((double)ks[0][v] + ks[1][v]) + ((double)ks[2][v] + ks[3][v]);
            qk[v] += ((double)qs[0][v] + qs[1][v]) + ((double)qs[2][v] + qs[3][v]);
        }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        if (MODE == 1) skk[4 * quad + v][c] = kk[v];
        sqk[4 * quad + v][c] = qk[v];
    }
    // (beyond the request's last token: beta = 0 and a decay of 1)
    const float* gate = gates + (size_t)(tok0 + min(c, nt - 1)) * 2 * heads + head;
    sb[quad][c] = c < nt ? gate[0] : 0.f;
    sg[quad][c] = c < nt ? gate[heads] : 1.f;
    shared_barrier();
    float* to = scratch + ((size_t)blockIdx.x * heads + head) * BlockPlaces<MODE>::FLOATS;
    const float beta = sb[quad][c];
    double d = 1.0, all = sg[quad][0];                      // D_ic, and G_i
#pragma unroll
    for (int i = 0; i < BL_T; ++i) {
        const double g = sg[quad][i];
        if (i > 0) all *= g;
        if (i > c) d *= g;
        const float p = i >= c ? (float)(sqk[i][c] * d * (MODE == 1 ? 1.0 : (double)beta)) : 0.f;
        if (live) to[BlockPlaces<MODE>::P + i * BL_T + c] = i > c ? p : 0.f;
        if (live && i == c) to[BlockPlaces<MODE>::PD + c] = p;
        if (MODE == 1) sl[quad][i][c] = i > c ? sb[quad][i] * skk[i][c] * d : 0.0;
        if (live && c == 0) to[BlockPlaces<MODE>::G + i] = (float)all;
    }
    if (live) to[BlockPlaces<MODE>::W + c] = (float)(MODE == 1 ? d : d * beta);
    if (MODE == 1) {
        if (live) to[BlockPlaces<MODE>::TD + c] = beta;
        shared_barrier();
        double x[BL_T];                                     // column c of the inverse, times beta_c
#pragma unroll
        for (int i = 0; i < BL_T; ++i) {
            double s = i == c ? (double)beta : 0.0;
#pragma unroll
            for (int l = 0; l < i; ++l) s -= sl[quad][i][l] * x[l];
            x[i] = i >= c ? s : 0.0;
            if (live) to[BlockPlaces<MODE>::T + i * BL_T + c] = i > c ? (float)x[i] : 0.f;
        }
    }
}

// sum_j m_ij r_j of a lane's rows i = 4 quad + v over j < i alone, number by number, with m as the matrix instruction's left operand (lane l: row l % 16, columns 4 (l / 16) and
// up): where a later token's row of r is an infinity or a NaN, which the instruction would multiply by the zeros above the diagonal.  (From registers: a load here would make
// the compiler wait for all that are on their way, on the usual path too.)
__device__ __forceinline__ bl_f32x4 bl_lower_product(bl_f32x4 m, bl_f32x4 r) {
    const int lane = threadIdx.x & 63, quad = lane >> 4, c = lane & 15;
    bl_f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int j = 0; j < BL_T; ++j) {
        const float rj = (j & 2) ? ((j & 1) ? r[3] : r[2]) : ((j & 1) ? r[1] : r[0]), mj = (j & 2) ? ((j & 1) ? m[3] : m[2]) : ((j & 1) ? m[1] : m[0]);
        const float x = __shfl(rj, (j >> 2) * 16 + c, TL_WAVE);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float y = __shfl(mj, (j >> 2) * 16 + 4 * quad + v, TL_WAVE);
            if (j < 4 * quad + v) s[v] = fmaf(y, x, s[v]);
        }
    }
    return s;
}

// MODE as the token loop's (1 or 2).  NT: a wave's rows in tiles of 16, 64 NT >= dim; WHOLE: 64 NT == dim.
template <int MODE, int NT, bool WHOLE>
__global__ void __launch_bounds__(320, NT <= 2 ? 3 : 2)
block_scan_kernel(const float* __restrict__ qkv, const float* __restrict__ scratch, const float* __restrict__ head_skip, float* __restrict__ state, size_t slot_stride,
                  const int* __restrict__ slots, const int* __restrict__ req_indptr, float* __restrict__ out, int heads, int kv_heads, int dim, int vdim, int least, int blocks) {
    __shared__ bl_f32x4 part[3][2][4][TL_WAVE];              // the waves' shares of K S and Q S, of three blocks in turn: at a barrier the fifth wave still reads those of the block before
    __shared__ bl_f32x4 su[2][TL_WAVE];                      // U
    typedef BlockPlaces<MODE> Places;
    // neighbouring heads, which share keys and queries, and all columns of a head on one XCD where that deals out evenly: what one work-group fetches the others find in its L2
    const int req = blockIdx.z, head = heads % 8 == 0 ? (int)(blockIdx.x % 8) * (heads / 8) + (int)blockIdx.x / 8 : (int)blockIdx.x;
    const int tok0 = req_indptr[req], tok1 = req_indptr[req + 1];
    if (tok1 - tok0 < least) return;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TL_WAVE), lane = threadIdx.x % TL_WAVE, quad = lane >> 4, c = lane & 15;
    int first = 0;
    for (int base = 0; base < req; base += TL_WAVE) {
        int mine = base + lane < req ? bl_blocks(req_indptr, base + lane, least) : 0;
#pragma unroll
        for (int o = TL_WAVE / 2; o > 0; o >>= 1) mine += __shfl_xor(mine, o, TL_WAVE);
        first += mine;
    }
    first = __builtin_amdgcn_readfirstlane(first);
    const int full = (tok1 - tok0) / BL_T, left = (tok1 - tok0) % BL_T;
    if (first + full + (left > 0) > blocks) return;        // (more than the caller counted: nothing is read beyond the scratch)
    const int C = 2 * kv_heads * dim + heads * vdim, kv = head / (heads / kv_heads), col = blockIdx.y * BL_T + c;
    const float* q_base = qkv + (size_t)tok0 * C + kv * dim;
    const float* k_base = q_base + kv_heads * dim;
    const float* v_base = qkv + (size_t)tok0 * C + 2 * kv_heads * dim + (size_t)head * vdim;
    const float* m_base = scratch + ((size_t)first * heads + head) * Places::FLOATS;
    float* o_base = out + ((size_t)tok0 * heads + head) * vdim;
    const int count = full + (left > 0);
    auto total = [&](int block, int which) {
        const bl_f32x4(&x)[4][TL_WAVE] = part[block % 3][which];
        return (x[0][lane] + x[1][lane]) + (x[2][lane] + x[3][lane]);
    };
    auto odd = [&](const bl_f32x4& x) {
        const float most = fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3])));
        const float sum = (x[0] + x[1]) + (x[2] + x[3]);   // (a maximum passes a NaN over, a sum does not)
        return __ballot(!(most <= 3.402823466e38f) || sum != sum) != 0;
    };

    if (wave == 4) {                                       // the outputs, a block behind the others
        const float skip = MODE == 2 ? head_skip[head] : 0.f;
        const unsigned value_at = (unsigned)min(col, vdim - 1);
        struct { bl_f32x4 P, Pd, G, value; } ops[4];       // of four blocks, each requested when its place is free
        auto fetch = [&](int place, int block) {
            const float* m = m_base + (size_t)block * heads * Places::FLOATS;
            ops[place].P = *(const bl_f32x4*)(m + Places::P + c * BL_T + 4 * quad);
            ops[place].Pd = *(const bl_f32x4*)(m + Places::PD + 4 * quad);
            ops[place].G = *(const bl_f32x4*)(m + Places::G + 4 * quad);
            if (MODE == 2) {
#pragma unroll
                for (int v = 0; v < 4; ++v) ops[place].value[v] = v_base[(size_t)min(block * BL_T + 4 * quad + v, tok1 - tok0 - 1) * C + value_at];
            }
        };
#pragma unroll
        for (int i = 0; i < 4; ++i) fetch(i, min(i, count - 1));
        shared_barrier();
        auto outputs = [&](int i, int block) {
            shared_barrier();                              // (the others' next block, or their end)
            bl_f32x4 u, before = total(block, 1);
            if (MODE == 1) u = su[block & 1][lane];
#pragma unroll
            for (int v = 0; v < 4; ++v) if (MODE == 2) u[v] = block * BL_T + 4 * quad + v < tok1 - tok0 ? ops[i].value[v] : 0.f;
            bl_f32x4 o = {0.f, 0.f, 0.f, 0.f};
            if (odd(u)) o = bl_lower_product(ops[i].P, u);
            else {
#pragma unroll
                for (int v = 0; v < 4; ++v) o = __builtin_amdgcn_mfma_f32_16x16x4f32(ops[i].P[v], u[v], o, 0, 0, 0);
            }
            float* to = o_base + (size_t)block * BL_T * heads * vdim;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float x = fmaf(ops[i].Pd[v], u[v], fmaf(ops[i].G[v], before[v], o[v]));
                if (col < vdim && block * BL_T + 4 * quad + v < tok1 - tok0) to[(unsigned)((4 * quad + v) * heads * vdim + col)] = MODE == 2 ? fmaf(skip, u[v], x) : x;
            }
            fetch(i, min(block + 4, count - 1));
        };
        int block = 0;
        for (; block + 3 < count; block += 4) {
#pragma unroll
            for (int i = 0; i < 4; ++i) outputs(i, block + i);
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
            if (block + i < count) outputs(i, block + i);
        return;
    }

    const int row0 = wave * 16 * NT;
    float* st = state + (size_t)slots[req] * slot_stride + (size_t)head * vdim * dim + (size_t)min(col, vdim - 1) * dim;
    bl_f32x4 S[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int r = row0 + 16 * t + 4 * quad;
        S[t] = bl_f32x4{0.f, 0.f, 0.f, 0.f};
        if (r < dim && col < vdim) S[t] = *(const bl_f32x4*)(st + r);
    }

    // A block's operands: keys and queries of token c as left operands of the products with S, keys of tokens 4 quad + v as that of the state's update, the block's matrices,
    // values.  They are requested two blocks ahead (a trip to memory takes as long as a block's work), by a base that the wave shares and offsets of the lane's
    // that never change and without a branch (behind one the compiler waits for every request on its way): rows beyond dim are copies, whose share of the state's update is
    // zeroed, and the blocks are whole; a request's last, broken one has a fetch of its own.
    struct Operands { bl_f32x4 k[NT], q[NT], T, G, w, Td; float kt[NT][4], v[4], all; } ops[2];
    unsigned row_at[NT], turned_at[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        row_at[t] = (unsigned)(c * C + (WHOLE ? row0 + 16 * t + 4 * quad : min(row0 + 16 * t + 4 * quad, dim - 4)));
        turned_at[t] = (unsigned)(4 * quad * C + (WHOLE ? row0 + 16 * t + c : min(row0 + 16 * t + c, dim - 1)));
    }
    const unsigned value_at = (unsigned)(4 * quad * C + min(col, vdim - 1));
    auto fetch_rows = [&](Operands& n, int block) {
        const float* kb = k_base + (size_t)block * BL_T * C;
        const float* qb = q_base + (size_t)block * BL_T * C;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if (MODE == 1) n.k[t] = *(const bl_f32x4*)(kb + row_at[t]);
            n.q[t] = *(const bl_f32x4*)(qb + row_at[t]);
        }
    };
    auto fetch_matrices = [&](Operands& n, int block) {
        const float* m = m_base + (size_t)block * heads * Places::FLOATS;
        if (MODE == 1) {
            n.G = *(const bl_f32x4*)(m + Places::G + 4 * quad);
            n.T = *(const bl_f32x4*)(m + Places::T + c * BL_T + 4 * quad);
            n.Td = *(const bl_f32x4*)(m + Places::TD + 4 * quad);
        }
        n.w = *(const bl_f32x4*)(m + Places::W + 4 * quad);
        n.all = m[Places::G + BL_T - 1];
    };
    auto fetch_rest = [&](Operands& n, int block) {
        const float* kb = k_base + (size_t)block * BL_T * C;
        const float* vb = v_base + (size_t)block * BL_T * C;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            n.v[v] = (vb + v * C)[value_at];
#pragma unroll
            for (int t = 0; t < NT; ++t) n.kt[t][v] = (kb + v * C)[turned_at[t]];
        }
        fetch_matrices(n, block);
    };
    auto fetch_broken = [&](Operands& n, int block) {       // `left` tokens; the others' keys, queries and values are zeros (and their step sizes)
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            n.k[t] = n.q[t] = bl_f32x4{0.f, 0.f, 0.f, 0.f};
            if (c < left) {
                if (MODE == 1) n.k[t] = *(const bl_f32x4*)(k_base + (size_t)block * BL_T * C + row_at[t]);
                n.q[t] = *(const bl_f32x4*)(q_base + (size_t)block * BL_T * C + row_at[t]);
            }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const bool in = 4 * quad + v < left;
            n.v[v] = in ? v_base[(size_t)(block * BL_T + v) * C + value_at] : 0.f;
#pragma unroll
            for (int t = 0; t < NT; ++t) n.kt[t][v] = in ? k_base[(size_t)(block * BL_T + v) * C + turned_at[t]] : 0.f;
        }
        fetch_matrices(n, block);
    };
    // ahead: the block to request next, whole; broken: whether this is the last block of `left` tokens, behind which nothing is requested
    auto work = [&](Operands& n, int block, int ahead, auto broken) {
        // K S, then Q S, four sums each; K S is exchanged while Q S is made
        bl_f32x4 a[4], b[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) a[v] = b[v] = bl_f32x4{0.f, 0.f, 0.f, 0.f};
        if (MODE == 1) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) a[v] = __builtin_amdgcn_mfma_f32_16x16x4f32(n.k[t][v], S[t][v], a[v], 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) b[v] = __builtin_amdgcn_mfma_f32_16x16x4f32(n.q[t][v], S[t][v], b[v], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        bl_f32x4(&shares)[2][4][TL_WAVE] = part[block % 3];
        if (MODE == 1) {
            shares[0][wave][lane] = (a[0] + a[1]) + (a[2] + a[3]);
            shared_barrier();
        }
        const bl_f32x4 value = {n.v[0], n.v[1], n.v[2], n.v[3]};
        bl_f32x4 u = value, r = value;
        if (MODE == 1) {
            const bl_f32x4 sum = total(block, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                r[v] = fmaf(-n.G[v], sum[v], value[v]);
                if (broken && 4 * quad + v >= left) r[v] = 0.f;
            }
            // (the diagonal's share, the largest, goes in last and once: in the matrix instruction every small one after it would be rounded at its size)
            u = bl_f32x4{0.f, 0.f, 0.f, 0.f};
            if (odd(r)) u = bl_lower_product(n.T, r);
            else {
#pragma unroll
                for (int v = 0; v < 4; ++v) u = __builtin_amdgcn_mfma_f32_16x16x4f32(n.T[v], r[v], u, 0, 0, 0);
            }
        }
        if (!broken) fetch_rows(n, ahead);
        shares[1][wave][lane] = (b[0] + b[1]) + (b[2] + b[3]);      // (for the fifth wave, behind the next barrier)
        if (MODE == 1) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                u[v] = fmaf(n.Td[v], r[v], u[v]);
                if (broken && 4 * quad + v >= left) u[v] = 0.f;
            }
            if (wave == 0) su[block & 1][lane] = u;
        }
        bl_f32x4 more[NT];                                  // (apart from S, which is rounded once a block)
#pragma unroll
        for (int t = 0; t < NT; ++t) more[t] = bl_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float wu = n.w[v] * u[v];
#pragma unroll
            for (int t = 0; t < NT; ++t)
                more[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(WHOLE || row0 + 16 * t + c < dim ? n.kt[t][v] : 0.f, wu, more[t], 0, 0, 0);
        }
        const float all = n.all;
        if (!broken) fetch_rest(n, ahead);
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) S[t][v] = fmaf(all, S[t][v], more[t][v]);
        if (MODE == 2) shared_barrier();
    };
    if (full > 0) {
        fetch_rows(ops[0], 0);
        fetch_rest(ops[0], 0);
        fetch_rows(ops[1], min(1, full - 1));
        fetch_rest(ops[1], min(1, full - 1));
    }
    int block = 0;
    for (; block + 1 < full; block += 2) {                  // (no way past one of the two: behind it the compiler would wait for what the other requests)
        work(ops[0], block, min(block + 2, full - 1), std::false_type{});
        work(ops[1], block + 1, min(block + 3, full - 1), std::false_type{});
    }
    if (block < full) work(ops[0], block, full - 1, std::false_type{});
    if (left > 0) {
        fetch_broken(ops[0], full);
        work(ops[0], full, full, std::true_type{});
    }
    shared_barrier();                                       // the last block's outputs
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int r = row0 + 16 * t + 4 * quad;
        if (r < dim && col < vdim) *(bl_f32x4*)(st + r) = S[t];
    }
}

// Numbers of scratch for so many blocks.
extern "C" long tl_blocks_floats(int mode, int blocks, int heads) { return (long)blocks * heads * (mode == 1 ? BlockPlaces<1>::FLOATS : BlockPlaces<2>::FLOATS); }

// Whether a step's long portions (`tokens` in all, the longest of so many) go through the blocks, beside `rest` requests of a few tokens: two estimates in us, fitted to both ways'
// times over 1600 steps of 128 to 9000 tokens at 2 to 128 heads and held against 600 others: the way it takes is 1.010 times the faster one's time on average, 13 of the 600 go through
// blocks that the loop would be more than 3 % ahead of, 26 stay with a loop more than 8 % behind.  The loop's and the blocks' time is a chain along the longest portion and, where the
// work-groups outnumber the chip, the work: about the same on both ways, but for the matrices, which the blocks cost more, so that the delta rule's steps of many thousand tokens in many
// portions stay with the loop.
// Measured (us, loop / blocks): the delta rule, 16 heads of 128 x 128: 128 tokens 27 / 22, 256 50 / 30, 512 106 / 48, 2048 413 / 162; 128 to 900 tokens of four requests 196 / 105,
// 16 x 128 102 / 109, 4 x 512 127 / 91, 64 x 128 351 / 420; 32 heads: 512 109 / 52, 16 x 128 178 / 206, 64 x 128 676 / 872, 32 x 256 666 / 776, 16 x 512 673 / 724; 4 heads of
// 64 x 64: 512 73 / 37; 8 heads of 256 x 256: 128 72 / 32, 512 291 / 76; the selective recurrence, 128 heads of 128 x 64: 128 28 / 21, 512 99 / 49, 16 x 128 241 / 213, 64 x 128 972 / 903.
extern "C" int tl_blocks_pay(int mode, int tokens, int longest, int rest, int heads, int dim, int vdim) {
    const double groups = (double)heads * ((vdim + BL_T - 1) / BL_T), rows = (dim + 63) / 64;
    const double work = tokens * groups * 256.0 / tl_mlstm_units * fmax(1.0, rows / 2);
    const double loop = 0.7 + hypot(longest * (rows > 3 ? 0.62 : 0.099 + 0.057 * rows), work * (mode == 1 ? 3.57e-4 : 2.55e-4));
    const double blocks = 10.3 + tokens * (double)heads * rows * (mode == 1 ? 3.35e-4 : 0.16e-4) + (rest > 0 ? 12 : 0) +
                          hypot(longest * (0.036 + 0.010 * rows), work * (rows > 1 ? 1.0 : 0.84) * (mode == 1 ? 2.73e-4 : 1.84e-4));
    return blocks < loop;
}

// Whether the requests of `least` tokens and more can go through the blocks: whole pieces of four numbers, and scratch for all of them.
static bool blocks_fit(int mode, const void* qkv, int heads, int kv_heads, int dim, int vdim, const void* state, long slot_stride, int blocks, const void* scratch, long floats) {
    return scratch && blocks > 0 && floats >= tl_blocks_floats(mode, blocks, heads) && dim % 4 == 0 && (2 * kv_heads * dim + heads * vdim) % 4 == 0 && ((uintptr_t)qkv & 15) == 0 &&
           ((uintptr_t)state & 15) == 0 && slot_stride % 4 == 0 && ((uintptr_t)scratch & 15) == 0 && (long)kv_heads * ((heads / kv_heads + 3) / 4) <= 65535;
}

template <int MODE>
static void launch_blocks(const void* qkv, const void* gates, const void* skip, void* state, long slot_stride, const void* slots, const void* req_indptr, void* out,
                          int requests, int heads, int kv_heads, int dim, int vdim, int least, int blocks, void* scratch, hipStream_t stream) {
    const dim3 mgrid(blocks, kv_heads * ((heads / kv_heads + 3) / 4)), grid(heads, (vdim + BL_T - 1) / BL_T, requests);
    block_matrices_kernel<MODE><<<mgrid, 64, 0, stream>>>((const float*)qkv, (const float*)gates, (const int*)req_indptr, (float*)scratch, requests, heads, kv_heads, dim, vdim, least);
#define TL_BLOCKS_W(N, W) block_scan_kernel<MODE, N, W><<<grid, 320, 0, stream>>>((const float*)qkv, (const float*)scratch, (const float*)skip, (float*)state, (size_t)slot_stride, \
        (const int*)slots, (const int*)req_indptr, (float*)out, heads, kv_heads, dim, vdim, least, blocks)
#define TL_BLOCKS(N) if (dim == 64 * N) TL_BLOCKS_W(N, true); else TL_BLOCKS_W(N, false)
    if (dim <= 64) { TL_BLOCKS(1); }
    else if (dim <= 128) { TL_BLOCKS(2); }
    else if (dim <= 192) { TL_BLOCKS(3); }
    else { TL_BLOCKS(4); }
#undef TL_BLOCKS_W
#undef TL_BLOCKS
}

// With scratch (null: the token loop alone) requests of at least `least` tokens go through the blocks where the rows allow it (`blocks`: no fewer than they make), and the
// token loop takes the others (rest: how many there are, or more if the caller cannot tell; 0 only if there are none), of about rest_longest tokens at most.
extern "C" int tl_delta_scan(const void* qkv, const void* gates, void* state, long slot_stride, const void* slots, const void* req_indptr,
                             void* out, int requests, int heads, int kv_heads, int dim, int vdim, int tokens, int longest, int least, int blocks, int rest,
                             int rest_longest, void* scratch, long scratch_floats, hipStream_t stream) {
    TL_REQUIRE(requests >= 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && vdim > 0, "delta_scan: bad sizes");
    TL_REQUIRE(dim <= DELTA_L * 16, "delta_scan: built for up to %d query/key dimensions per head, got %d", DELTA_L * 16, dim);
    TL_REQUIRE(slot_stride >= (long)heads * dim * vdim, "delta_scan: the state rows are too short");
    TL_REQUIRE(requests <= 65535 && heads <= 65535, "delta_scan: too many requests or heads for one launch");
    if (requests == 0) return TL_OK;
    const bool through = blocks_fit(1, qkv, heads, kv_heads, dim, vdim, state, slot_stride, blocks, scratch, scratch_floats);
    if (through) {
        launch_blocks<1>(qkv, gates, nullptr, state, slot_stride, slots, req_indptr, out, requests, heads, kv_heads, dim, vdim, least, blocks, scratch, stream);
        TL_CHECK_LAUNCH("delta_blocks");
        if (rest == 0) return TL_OK;
    }
    launch_delta_scan<1>(qkv, gates, nullptr, state, slot_stride, slots, req_indptr, out, requests, heads, kv_heads, dim, vdim, through ? rest * rest_longest : tokens,
                         through ? rest_longest : longest, through ? least : INT_MAX, stream);
    TL_CHECK_LAUNCH("delta_scan");
    return TL_OK;
}

// ------------------------------------------------------------------ what the selective state-space recurrence reads
// Made from the projection of the step's tokens.  proj [T, ld] holds per token, from column x_off on, the
// `channels` = inner + 2 * groups * state convolved channels [x | B | C] and after them `heads` raw step sizes.  Channel c at the request's
// i-th token of the step: y = silu(bias[c] + sum_j w[c][j] * in[i - (taps - 1) + j][c]) with in[i'] the projection of the step's token
// i' >= 0, else tail[taps - 1 + i'][c] (the slot's last taps - 1 inputs from before the step; zero for a new request).  y goes to qkv
// float [T, channels] in the order the recurrence reads: C, B, x.  gates float [T, 2 * heads] receives dt = softplus(raw + dt_bias) and
// decay = exp(-exp(a_log) * dt).  One thread per token and channel (or head).
template <typename T>
__global__ void __launch_bounds__(256)
selective_prepare_kernel(const T* __restrict__ proj, int ld, int x_off, const float* __restrict__ conv_w, const float* __restrict__ conv_b,
                         float* __restrict__ gates, const float* __restrict__ a_log, const float* __restrict__ dt_bias,
                         const float* __restrict__ state, size_t slot_stride, size_t tail_off, const int* __restrict__ slots,
                         const int* __restrict__ req_indptr, const int* __restrict__ token_req, float* __restrict__ qkv, int heads, int inner,
                         int gn, int taps) {
    const int t = blockIdx.x, c = blockIdx.y * blockDim.x + threadIdx.x;
    const int channels = inner + 2 * gn;
    if (c >= channels + heads) return;
    const T* row = proj + (size_t)t * ld + x_off;
    if (c >= channels) {
        const int h = c - channels;
        const float dt = softplus_f(to_float(row[c]) + dt_bias[h]);
        gates[(size_t)t * 2 * heads + h] = dt;
        gates[(size_t)t * 2 * heads + heads + h] = expf(-expf(a_log[h]) * dt);
        return;
    }
    const int req = token_req[t];
    const int i = t - req_indptr[req];
    const float* tail = state + (size_t)slots[req] * slot_stride + tail_off;
    float acc = conv_b[c];
    for (int j = 0; j < taps; ++j) {
        const int back = i - (taps - 1) + j;
        const float xv = back >= 0 ? to_float(proj[(size_t)(t - i + back) * ld + x_off + c]) : tail[(size_t)(taps - 1 + back) * channels + c];
        acc = fmaf(conv_w[(size_t)c * taps + j], xv, acc);
    }
    const int to = c < inner ? 2 * gn + c : (c < inner + gn ? gn + (c - inner) : c - inner - gn);
    qkv[(size_t)t * channels + to] = silu_f(acc);
}

extern "C" int tl_selective_prepare(const void* proj, int ld, int x_off, const void* conv_w, const void* conv_b, void* gates, const void* a_log,
                                    const void* dt_bias, void* state, long slot_stride, long tail_off, const void* slots, const void* req_indptr,
                                    const void* token_req, void* qkv, int tokens, int requests, int heads, int inner, int gn, int taps, int dtype,
                                    hipStream_t stream) {
    TL_REQUIRE(tokens >= 0 && requests >= 0 && heads > 0 && inner > 0 && gn > 0 && x_off >= 0, "selective_prepare: bad sizes");
    TL_REQUIRE(taps >= 1 && taps <= DELTA_MAX_TAPS, "selective_prepare: 1 to %d taps are built, not %d", DELTA_MAX_TAPS, taps);
    const int channels = inner + 2 * gn;
    TL_REQUIRE(ld >= x_off + channels + heads && tail_off >= 0 && slot_stride >= tail_off + (long)(taps - 1) * channels, "selective_prepare: rows or state too short");
    TL_REQUIRE(dtype == TL_DT_F32 || dtype == TL_DT_BF16, "selective_prepare: unknown dtype %d", dtype);
    TL_REQUIRE(requests <= 65535 && (channels + heads + 255) / 256 <= 65535, "selective_prepare: too many requests or channels for one launch");
    if (tokens == 0 || requests == 0) return TL_OK;
    dim3 grid(tokens, (channels + heads + 255) / 256), block(256);
    dim3 tgrid((channels + 255) / 256, requests), tblock(256);
    if (taps == 4 && conv_b) {
        ConvArgs a = {(const float*)conv_w, (const float*)conv_b, (float*)gates, (const float*)a_log, (const float*)dt_bias, (float*)state, (size_t)slot_stride,
                      (size_t)tail_off, (const int*)slots, (const int*)req_indptr, (const int*)token_req, (float*)qkv, ld, channels, tokens, heads,
                      0, 0, 1, 1.f, 0.f, inner, gn};
        bool tail_done = false;
        if (dtype == TL_DT_F32 ? short_conv<float, 1>((const float*)proj + x_off, a, requests, stream, &tail_done)
                               : short_conv<bf16_t, 1>((const bf16_t*)proj + x_off, a, requests, stream, &tail_done)) {
            TL_CHECK_LAUNCH("selective_prepare");
            if (tail_done) return TL_OK;
            if (dtype == TL_DT_F32) delta_tail_kernel<float><<<tgrid, tblock, 0, stream>>>((const float*)proj + x_off, ld, (float*)state, (size_t)slot_stride,
                                                                                           (size_t)tail_off, (const int*)slots, (const int*)req_indptr, channels, taps);
            else delta_tail_kernel<bf16_t><<<tgrid, tblock, 0, stream>>>((const bf16_t*)proj + x_off, ld, (float*)state, (size_t)slot_stride,
                                                                         (size_t)tail_off, (const int*)slots, (const int*)req_indptr, channels, taps);
            TL_CHECK_LAUNCH("selective_tail");
            return TL_OK;
        }
    }
#define TL_SP(T)                                                                                                                                  \
    selective_prepare_kernel<T><<<grid, block, 0, stream>>>((const T*)proj, ld, x_off, (const float*)conv_w, (const float*)conv_b, (float*)gates,     \
        (const float*)a_log, (const float*)dt_bias, (const float*)state, (size_t)slot_stride, (size_t)tail_off, (const int*)slots,               \
        (const int*)req_indptr, (const int*)token_req, (float*)qkv, heads, inner, gn, taps);                                                      \
    TL_CHECK_LAUNCH("selective_prepare");                                                                                                         \
    if (taps > 1) delta_tail_kernel<T><<<tgrid, tblock, 0, stream>>>((const T*)proj + x_off, ld, (float*)state, (size_t)slot_stride, (size_t)tail_off, \
                                                                     (const int*)slots, (const int*)req_indptr, channels, taps)
    if (dtype == TL_DT_F32) { TL_SP(float); } else { TL_SP(bf16_t); }
#undef TL_SP
    TL_CHECK_LAUNCH("selective_tail");
    return TL_OK;
}

// out[t, c] = silu(float(x[t, c])) for the first `cols` columns of every row (the rows of x may be longer).
template <typename T>
__global__ void silu_float_kernel(const T* __restrict__ x, int ld, float* __restrict__ out, int cols, size_t total) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total) return;
    const float v = to_float(x[(i / cols) * ld + i % cols]);
    out[i] = v / (1.f + expf(-v));
}

extern "C" int tl_silu_float(const void* x, int ld, void* out, int rows, int cols, int dtype, hipStream_t stream) {
    TL_REQUIRE(rows >= 0 && cols > 0 && ld >= cols, "silu_float: bad sizes");
    if (rows == 0) return TL_OK;
    const size_t total = (size_t)rows * cols;
    const int grid = (int)((total + 255) / 256);
    if (dtype == TL_DT_F32) silu_float_kernel<float><<<grid, 256, 0, stream>>>((const float*)x, ld, (float*)out, cols, total);
    else if (dtype == TL_DT_BF16) silu_float_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)x, ld, (float*)out, cols, total);
    else TL_REQUIRE(false, "silu_float: unknown dtype %d", dtype);
    TL_CHECK_LAUNCH("silu_float");
    return TL_OK;
}

// ------------------------------------------------------------------ decays per key channel
// decay[t, n] = exp(-exp(w0[n] + sum_j w2t[j][n] * tanh(z[t, j]))): z float [tokens, rank], w2t float [rank][channels].  A work-group of 256
// threads takes 256 channels of TT tokens, a thread a channel; the order of a sum does not depend on TT.
template <int TT>
__global__ void __launch_bounds__(256)
channel_decay_kernel(const float* __restrict__ z, const float* __restrict__ w2t, const float* __restrict__ w0, float* __restrict__ decay,
                     int tokens, int rank, int channels) {
    extern __shared__ __attribute__((aligned(16))) float cd_tanh[];          // [rank][TT]
    const int t0 = blockIdx.y * TT, n = blockIdx.x * 256 + threadIdx.x;
    for (int i = threadIdx.x; i < rank * TT; i += 256) {
        const int tt = i / rank, j = i % rank;
        cd_tanh[j * TT + tt] = t0 + tt < tokens ? tanhf(z[(size_t)(t0 + tt) * rank + j]) : 0.f;
    }
    __syncthreads();
    if (n >= channels) return;
    float acc[TT];
    const float start = w0[n];
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) acc[tt] = start;
#pragma unroll 8
    for (int j = 0; j < rank; ++j) {
        const float w = w2t[(size_t)j * channels + n];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) acc[tt] = fmaf(w, cd_tanh[j * TT + tt], acc[tt]);
    }
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
        if (t0 + tt < tokens) decay[(size_t)(t0 + tt) * channels + n] = expf(-expf(acc[tt]));
}

extern "C" int tl_channel_decay(const void* z, const void* w2t, const void* w0, void* decay, int tokens, int rank, int channels, hipStream_t stream) {
    TL_REQUIRE(tokens >= 0 && rank > 0 && channels > 0, "channel_decay: bad sizes");
    TL_REQUIRE(rank <= 1024, "channel_decay: built for ranks up to 1024, got %d", rank);
    if (tokens == 0) return TL_OK;
    const int blocks = (channels + 255) / 256;
    if ((long)blocks * tokens <= 1024)
        channel_decay_kernel<1><<<dim3(blocks, tokens), 256, sizeof(float) * rank, stream>>>((const float*)z, (const float*)w2t, (const float*)w0, (float*)decay, tokens, rank, channels);
    else
        channel_decay_kernel<8><<<dim3(blocks, (tokens + 7) / 8), 256, sizeof(float) * 8 * rank, stream>>>((const float*)z, (const float*)w2t, (const float*)w0, (float*)decay, tokens, rank, channels);
    TL_CHECK_LAUNCH("channel_decay");
    return TL_OK;
}

// ------------------------------------------------------------------ the recurrence with decays per key channel and a bonus
// Per request and head a state S of dim x vdim numbers; per token, with r, k (dim), v (vdim), the decays w (dim) and the head's bonus u (dim):
//   o = (S + diag(u) k v^T)^T r,   then   S <- diag(w) S + k v^T.
// Column j of S needs only its own sum_i r[i] S[i][j] and the number sum_i r[i] u[i] k[i], which all columns of the head share and which is
// made once per token.  The 16 lanes of a row of the wave share a column: lane i owns the rows 64 q + 4 i .. + 3 (q < RPL / 4) of it in
// registers for all tokens of the step, so the lanes' pieces of r, k and w lie side by side in shared memory and those of the state side by
// side in memory ([vdim][dim] per head).  Nothing but S itself passes from token to token: the sums over the lanes leave the chain.  A wave
// has 4 columns, a work-group of four waves 16.  The order of every sum is fixed by dim, so a token's result depends neither on how its
// request was cut into steps nor on what else the step holds.  Tokens are taken TB at a time (1, 4 or 16, by the longest portion of the
// step), fetched into registers one batch ahead; a request's last batch is filled up with tokens that change nothing (k = 0, w = 1).
// `last_rows` (optional, float [tokens, row_width]): the row of the request's last token goes to its slot from tail_off on (what the next
// portion's first token finds of the token before it).

template <typename T, int RPL, int TB>
__global__ void __launch_bounds__(256)
wkv_scan_kernel(const T* __restrict__ rkv, int ld, int k_off, int v_off, const float* __restrict__ decay, const float* __restrict__ bonus,
                float* __restrict__ state, size_t slot_stride, const int* __restrict__ slots, const int* __restrict__ req_indptr,
                float* __restrict__ out, int heads, int dim, int vdim, int vec, const float* __restrict__ last_rows, int row_width, size_t tail_off) {
    constexpr int ROWS = DELTA_L * RPL, Q = RPL / 4;            // ROWS >= dim
    constexpr int PPT = ROWS / 4, PIECES = TB * PPT, NP = (PIECES + 255) / 256;      // pieces of four numbers: per token, per batch, per thread
    __shared__ __attribute__((aligned(16))) float sr[TB * ROWS], sk[TB * ROWS], sw[TB * ROWS];
    __shared__ float sv[TB * DELTA_COLS], sb[TB];
    const int req = blockIdx.z, head = blockIdx.y, col0 = blockIdx.x * DELTA_COLS;
    const int tok0 = req_indptr[req], tok1 = req_indptr[req + 1];
    if (tok0 >= tok1) return;
    const int tid = threadIdx.x, wave = tid / TL_WAVE, lane = tid % TL_WAVE;
    const int rg = lane & 15, cw = wave * 4 + (lane >> 4);       // the lane's place in its column, and the column within the work-group
    const int col = col0 + cw;
    const bool col_ok = col < vdim;
    float* slot = state + (size_t)slots[req] * slot_stride;
    float* st = slot + ((size_t)head * vdim + col) * dim;

    float S[RPL], ub[RPL];
    const bool vec_state = vec && ((uintptr_t)state & 15) == 0 && (slot_stride & 3) == 0;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int row = 64 * q + 4 * rg;
        if (vec_state && col_ok && row + 4 <= dim) {
            const float4 x = *(const float4*)(st + row);
            S[4 * q] = x.x; S[4 * q + 1] = x.y; S[4 * q + 2] = x.z; S[4 * q + 3] = x.w;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) S[4 * q + e] = (col_ok && row + e < dim) ? st[row + e] : 0.f;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) ub[4 * q + e] = row + e < dim ? bonus[head * dim + row + e] : 0.f;
    }

    float4 pr[NP], pk[NP], pw[NP];
    float pv = 0.f;
    auto fetch = [&](int base) {
        const int nb = min(TB, tok1 - base);
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const int idx = tid + j * 256, t = idx / PPT, e = (idx % PPT) * 4;
            pr[j] = pk[j] = make_float4(0.f, 0.f, 0.f, 0.f);
            pw[j] = make_float4(1.f, 1.f, 1.f, 1.f);
            if (idx < PIECES && t < nb && e < dim) {
                const T* row = rkv + (size_t)(base + t) * ld + head * dim + e;
                const float* wrow = decay + ((size_t)(base + t) * heads + head) * dim + e;
                if (vec) {
                    pr[j] = load4(row);
                    pk[j] = load4(row + k_off);
                    pw[j] = *(const float4*)wrow;
                } else {
                    float a[4], b[4], c[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const bool ok = e + u < dim;
                        a[u] = ok ? to_float(row[u]) : 0.f;
                        b[u] = ok ? to_float(row[k_off + u]) : 0.f;
                        c[u] = ok ? wrow[u] : 1.f;
                    }
                    pr[j] = make_float4(a[0], a[1], a[2], a[3]);
                    pk[j] = make_float4(b[0], b[1], b[2], b[3]);
                    pw[j] = make_float4(c[0], c[1], c[2], c[3]);
                }
            }
        }
        if (tid < TB * DELTA_COLS) {
            const int t = tid / DELTA_COLS, c = tid % DELTA_COLS;
            pv = (t < nb && col0 + c < vdim) ? to_float(rkv[(size_t)(base + t) * ld + v_off + head * vdim + col0 + c]) : 0.f;
        }
    };
    fetch(tok0);
    for (int base = tok0; base < tok1; base += TB) {
        const int nb = min(TB, tok1 - base);
        shared_barrier();                              // the batch before has been worked on
#pragma unroll
        for (int j = 0; j < NP; ++j) {
            const int idx = tid + j * 256;
            if (idx < PIECES) {
                *(float4*)(sr + idx * 4) = pr[j];
                *(float4*)(sk + idx * 4) = pk[j];
                *(float4*)(sw + idx * 4) = pw[j];
            }
        }
        if (tid < TB * DELTA_COLS) sv[tid] = pv;
        if (base + TB < tok1) fetch(base + TB);
        shared_barrier();
        // the bonus sums: the 16 lanes of column cw make token cw's
        if (cw < TB) {
            float b4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const float4 k4 = *(const float4*)(sk + cw * ROWS + 64 * q + 4 * rg), r4 = *(const float4*)(sr + cw * ROWS + 64 * q + 4 * rg);
                b4[0] = fmaf(k4.x * ub[4 * q], r4.x, b4[0]);
                b4[1] = fmaf(k4.y * ub[4 * q + 1], r4.y, b4[1]);
                b4[2] = fmaf(k4.z * ub[4 * q + 2], r4.z, b4[2]);
                b4[3] = fmaf(k4.w * ub[4 * q + 3], r4.w, b4[3]);
            }
            const float b = row16_sum((b4[0] + b4[1]) + (b4[2] + b4[3]));
            if (rg == 0) sb[cw] = b;
        }
        shared_barrier();
        float mine = 0.f;                              // the output of token rg of the batch
#pragma unroll 4
        for (int t = 0; t < TB; ++t) {
            const float vt = sv[t * DELTA_COLS + cw];
            float o4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const int at = t * ROWS + 64 * q + 4 * rg;
                const float4 r4 = *(const float4*)(sr + at), k4 = *(const float4*)(sk + at), w4 = *(const float4*)(sw + at);
                o4[0] = fmaf(r4.x, S[4 * q], o4[0]);
                o4[1] = fmaf(r4.y, S[4 * q + 1], o4[1]);
                o4[2] = fmaf(r4.z, S[4 * q + 2], o4[2]);
                o4[3] = fmaf(r4.w, S[4 * q + 3], o4[3]);
                S[4 * q] = fmaf(w4.x, S[4 * q], k4.x * vt);
                S[4 * q + 1] = fmaf(w4.y, S[4 * q + 1], k4.y * vt);
                S[4 * q + 2] = fmaf(w4.z, S[4 * q + 2], k4.z * vt);
                S[4 * q + 3] = fmaf(w4.w, S[4 * q + 3], k4.w * vt);
            }
            const float o = fmaf(sb[t], vt, row16_sum((o4[0] + o4[1]) + (o4[2] + o4[3])));
            if (rg == t) mine = o;
        }
        if (rg < nb && col_ok) out[((size_t)(base + rg) * heads + head) * vdim + col] = mine;
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int row = 64 * q + 4 * rg;
        if (vec_state && col_ok && row + 4 <= dim) *(float4*)(st + row) = make_float4(S[4 * q], S[4 * q + 1], S[4 * q + 2], S[4 * q + 3]);
        else if (col_ok) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (row + e < dim) st[row + e] = S[4 * q + e];
        }
    }
    if (last_rows && blockIdx.x == 0) {                // the heads' first work-groups share the row
        for (int i = head * 256 + tid; i < row_width; i += heads * 256) slot[tail_off + i] = last_rows[(size_t)(tok1 - 1) * row_width + i];
    }
}

template <typename T>
static void launch_wkv_scan(const void* rkv, int ld, int k_off, int v_off, const void* decay, const void* bonus, void* state, long slot_stride,
                            const void* slots, const void* req_indptr, void* out, int requests, int heads, int dim, int vdim, int longest,
                            const void* last_rows, int row_width, long tail_off, hipStream_t stream) {
    const int rpl = dim <= 64 ? 4 : dim <= 128 ? 8 : dim <= 192 ? 12 : 16;
    const int tb = longest <= 1 ? 1 : (longest <= 4 ? 4 : DELTA_TB);
    const int vec = dim % 4 == 0 && ld % 4 == 0 && k_off % 4 == 0 && ((uintptr_t)rkv % (4 * sizeof(T))) == 0 && ((uintptr_t)decay & 15) == 0;
    dim3 grid((vdim + DELTA_COLS - 1) / DELTA_COLS, heads, requests), block(256);
#define TL_WKV_B(R, B)                                                                                                                       \
    wkv_scan_kernel<T, R, B><<<grid, block, 0, stream>>>((const T*)rkv, ld, k_off, v_off, (const float*)decay, (const float*)bonus, (float*)state, \
        (size_t)slot_stride, (const int*)slots, (const int*)req_indptr, (float*)out, heads, dim, vdim, vec, (const float*)last_rows, row_width, (size_t)tail_off)
#define TL_WKV(R)                        \
    if (tb == 1) TL_WKV_B(R, 1);         \
    else if (tb == 4) TL_WKV_B(R, 4);    \
    else TL_WKV_B(R, DELTA_TB)
    if (rpl == 4) { TL_WKV(4); }
    else if (rpl == 8) { TL_WKV(8); }
    else if (rpl == 12) { TL_WKV(12); }
    else { TL_WKV(16); }
#undef TL_WKV
#undef TL_WKV_B
}

// rkv [tokens, ld]: r of all heads at column 0 (heads * dim), k at k_off, v at v_off (heads * vdim); decay float [tokens, heads * dim]; bonus
// float [heads * dim]; the state of a head column by column ([vdim][dim]) from head * dim * vdim on in its slot; out float [tokens, heads * vdim].
extern "C" int tl_wkv_scan(const void* rkv, int ld, int k_off, int v_off, const void* decay, const void* bonus, void* state, long slot_stride,
                           const void* slots, const void* req_indptr, void* out, int requests, int heads, int dim, int vdim, int longest,
                           const void* last_rows, int row_width, long tail_off, int dtype, hipStream_t stream) {
    TL_REQUIRE(requests >= 0 && heads > 0 && dim > 0 && vdim > 0 && ld > 0 && k_off >= 0 && v_off >= 0, "wkv_scan: bad sizes");
    TL_REQUIRE(dim <= DELTA_L * 16, "wkv_scan: built for up to %d key dimensions per head, got %d", DELTA_L * 16, dim);
    TL_REQUIRE(slot_stride >= (long)heads * dim * vdim, "wkv_scan: the state rows are too short");
    TL_REQUIRE(!last_rows || (row_width > 0 && tail_off >= (long)heads * dim * vdim && slot_stride >= tail_off + row_width),
               "wkv_scan: the slots do not hold a row of %d numbers behind the states", row_width);
    TL_REQUIRE(requests <= 65535 && heads <= 65535, "wkv_scan: too many requests or heads for one launch");
    if (requests == 0) return TL_OK;
    if (dtype == TL_DT_F32) launch_wkv_scan<float>(rkv, ld, k_off, v_off, decay, bonus, state, slot_stride, slots, req_indptr, out, requests, heads, dim, vdim, longest, last_rows, row_width, tail_off, stream);
    else if (dtype == TL_DT_BF16) launch_wkv_scan<bf16_t>(rkv, ld, k_off, v_off, decay, bonus, state, slot_stride, slots, req_indptr, out, requests, heads, dim, vdim, longest, last_rows, row_width, tail_off, stream);
    else TL_REQUIRE(false, "wkv_scan: unknown dtype %d", dtype);
    TL_CHECK_LAUNCH("wkv_scan");
    return TL_OK;
}

// The same with what stands before and behind it, for steps of one token a request: the decays are made from their low-rank sums (channel_decay above), and the output goes through the norm of its
// head and the gate (gated_head_norm) before it is stored, all in the sums' order there.  A work-group has a whole head of a request: sixteen lanes a column and CG columns to each, whose states
// are all requested at the start, beside the token's numbers and the matrix of the decays; what a step waits for is then one trip to the state and the chain of tanh, the 64 products of a decay, the
// recurrence and the norm.  In three launches (decays, scan by four work-groups a head, norm) 16 requests with 32 heads of 64 x 64 took 6.8 + 9.2 + 4.1 us, in one 11.9.  Work-groups hold
// dim x vdim numbers of state, up to 128 x 128, in 169 to 272 registers: two of them share a compute unit, or none, and where more than a round or two of those queue the three launches, which deal a
// head's columns to several, are the faster ones (a decode step's call, 16 requests 6.8 us less in one launch, 32 0.8 less, 64 6.0 more).
template <typename T, int RPL, int CG>
__global__ void __launch_bounds__(256)
wkv_token_kernel(const T* __restrict__ rkv, int ld, int k_off, int v_off, int gate_off, const float* __restrict__ z, const float* __restrict__ w2t, const float* __restrict__ w0, int rank,
                 const float* __restrict__ bonus, float* __restrict__ state, size_t slot_stride, const int* __restrict__ slots, const int* __restrict__ req_indptr,
                 const float* __restrict__ norm, float eps, T* __restrict__ out, int heads, int dim, int vdim, const float* __restrict__ last_rows, int row_width, size_t tail_off) {
    constexpr int ROWS = DELTA_L * RPL, Q = RPL / 4, AHEAD = 64, LANES = CG <= 4 ? 16 : 32;
    __shared__ __attribute__((aligned(16))) float sr[ROWS], sk[ROWS], sw[ROWS], so[CG * 16];
    extern __shared__ __attribute__((aligned(16))) float wt_tanh[];          // [rank]
    const int req = blockIdx.y, head = blockIdx.x;
    const int slot_at = slots[req], tok0 = req_indptr[req], tok1 = req_indptr[req + 1];
    if (tok0 >= tok1) return;
    const int tid = threadIdx.x, wave = tid / TL_WAVE, lane = tid % TL_WAVE;
    const int rg = lane & 15, cw = wave * 4 + (lane >> 4);       // the lane's place in its columns, and the first of them
    const int channels = heads * dim, n = head * dim + min(tid, dim - 1);
    float* slot = state + (size_t)slot_at * slot_stride;
    float* st = slot + (size_t)head * vdim * dim;
    float S[CG][RPL];
#pragma unroll
    for (int c = 0; c < CG; ++c)
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int row = 64 * q + 4 * rg, col = 16 * c + cw;
            const float4 x = col < vdim && row < dim ? *(const float4*)(st + (size_t)col * dim + row) : make_float4(0.f, 0.f, 0.f, 0.f);
            S[c][4 * q] = x.x; S[c][4 * q + 1] = x.y; S[c][4 * q + 2] = x.z; S[c][4 * q + 3] = x.w;
        }
    float ub[RPL], ahead[AHEAD];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int row = 64 * q + 4 * rg;
        const float4 x = row < dim ? *(const float4*)(bonus + head * dim + row) : make_float4(0.f, 0.f, 0.f, 0.f);
        ub[4 * q] = x.x; ub[4 * q + 1] = x.y; ub[4 * q + 2] = x.z; ub[4 * q + 3] = x.w;
    }
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) ahead[j] = w2t[(size_t)min(j, rank - 1) * channels + n];
    const float start = w0[n];
    for (int t = tok0; t < tok1; ++t) {
        const T* row = rkv + (size_t)t * ld;
        if (tid < ROWS / 4) {
            const bool ok = 4 * tid < dim;
            *(float4*)(sr + 4 * tid) = ok ? load4(row + head * dim + 4 * tid) : make_float4(0.f, 0.f, 0.f, 0.f);
            *(float4*)(sk + 4 * tid) = ok ? load4(row + k_off + head * dim + 4 * tid) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        if (tid < ROWS) sw[tid] = 1.f;
        T v[CG];
#pragma unroll
        for (int c = 0; c < CG; ++c) v[c] = row[v_off + head * vdim + min(16 * c + cw, vdim - 1)];
        const int g_at = min(4 * (tid % LANES), vdim - 4);
        const typename Four<T>::type gate = *(const typename Four<T>::type*)(row + gate_off + head * vdim + g_at);
        const float4 nw = *(const float4*)(norm + head * vdim + g_at);
        for (int j = tid; j < rank; j += 256) wt_tanh[j] = tanhf(z[(size_t)t * rank + j]);
        __syncthreads();
        if (tid < dim) {
            float a = start;
#pragma unroll
            for (int j = 0; j < AHEAD; ++j)
                if (j < rank) a = fmaf(ahead[j], wt_tanh[j], a);
#pragma unroll 16
            for (int j = AHEAD; j < rank; ++j) a = fmaf(w2t[(size_t)j * channels + n], wt_tanh[j], a);
            sw[tid] = expf(-expf(a));
        }
        __syncthreads();
        float4 r4[Q], k4[Q], w4[Q];
        float b4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int at = 64 * q + 4 * rg;
            r4[q] = *(const float4*)(sr + at);
            k4[q] = *(const float4*)(sk + at);
            w4[q] = *(const float4*)(sw + at);
            b4[0] = fmaf(k4[q].x * ub[4 * q], r4[q].x, b4[0]);
            b4[1] = fmaf(k4[q].y * ub[4 * q + 1], r4[q].y, b4[1]);
            b4[2] = fmaf(k4[q].z * ub[4 * q + 2], r4[q].z, b4[2]);
            b4[3] = fmaf(k4[q].w * ub[4 * q + 3], r4[q].w, b4[3]);
        }
        const float b = row16_sum((b4[0] + b4[1]) + (b4[2] + b4[3]));
#pragma unroll
        for (int c = 0; c < CG; ++c) {
            const float vt = to_float(v[c]);
            float o4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                float* s4 = S[c] + 4 * q;
                o4[0] = fmaf(r4[q].x, s4[0], o4[0]);
                o4[1] = fmaf(r4[q].y, s4[1], o4[1]);
                o4[2] = fmaf(r4[q].z, s4[2], o4[2]);
                o4[3] = fmaf(r4[q].w, s4[3], o4[3]);
                s4[0] = fmaf(w4[q].x, s4[0], k4[q].x * vt);
                s4[1] = fmaf(w4[q].y, s4[1], k4[q].y * vt);
                s4[2] = fmaf(w4[q].z, s4[2], k4[q].z * vt);
                s4[3] = fmaf(w4[q].w, s4[3], k4[q].w * vt);
            }
            const float o = fmaf(b, vt, row16_sum((o4[0] + o4[1]) + (o4[2] + o4[3])));
            if (rg == 0) so[16 * c + cw] = o;
        }
        __syncthreads();
        if (wave == 0) {                                // the norm of the head and its gate, LANES lanes (the others do the same again and store nothing)
            const float4 u = *(const float4*)(so + g_at), g = widen4(gate);
            float ss = 0.f;
            if (4 * (lane % LANES) < vdim) { ss = fmaf(u.x, u.x, ss); ss = fmaf(u.y, u.y, ss); ss = fmaf(u.z, u.z, ss); ss = fmaf(u.w, u.w, ss); }
            const float inv = 1.f / sqrtf(lanes_sum<LANES>(ss) / (float)vdim + eps);
            const float4 s = make_float4(1.f / (1.f + expf(-g.x)), 1.f / (1.f + expf(-g.y)), 1.f / (1.f + expf(-g.z)), 1.f / (1.f + expf(-g.w)));
            if (4 * lane < vdim)
                store4(out + ((size_t)t * heads + head) * vdim + 4 * lane, make_float4(u.x * (g.x * s.x) * inv * nw.x, u.y * (g.y * s.y) * inv * nw.y,
                                                                                       u.z * (g.z * s.z) * inv * nw.z, u.w * (g.w * s.w) * inv * nw.w));
        }
        if (t + 1 < tok1) __syncthreads();              // (a request that brings more: its next token's numbers go where these were)
    }
#pragma unroll
    for (int c = 0; c < CG; ++c)
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int row = 64 * q + 4 * rg, col = 16 * c + cw;
            if (col < vdim && row < dim) *(float4*)(st + (size_t)col * dim + row) = make_float4(S[c][4 * q], S[c][4 * q + 1], S[c][4 * q + 2], S[c][4 * q + 3]);
        }
    if (last_rows)                                      // the heads share the row
        for (int i = head * 256 + tid; i < row_width; i += heads * 256) slot[tail_off + i] = last_rows[(size_t)(tok1 - 1) * row_width + i];
}

// Whether wkv_token_kernel is built for these sizes and places: heads in whole pieces of four numbers, on the places where they can be fetched.
extern "C" int tl_wkv_token_fits(const void* rkv, int ld, int k_off, int v_off, int gate_off, const void* bonus, const void* state, long slot_stride, const void* norm, const void* out, int dim,
                                 int vdim, int rank, int dtype) {
    const size_t piece = dtype == TL_DT_F32 ? 16 : 8;
    return (dtype == TL_DT_F32 || dtype == TL_DT_BF16) && dim > 0 && vdim > 0 && dim % 4 == 0 && vdim % 4 == 0 && dim <= 128 && vdim <= 128 && rank > 0 && rank <= 1024 &&
           (ld | k_off | v_off | gate_off) % 4 == 0 && slot_stride % 4 == 0 && ((uintptr_t)rkv | (uintptr_t)out) % piece == 0 && ((uintptr_t)bonus | (uintptr_t)state | (uintptr_t)norm) % 16 == 0;
}

// Operands as tl_wkv_scan and tl_channel_decay take them; the gate's numbers lie in the rows of rkv from gate_off on; norm float [heads * vdim]; out [tokens, heads * vdim] of rkv's type.
extern "C" int tl_wkv_token(const void* rkv, int ld, int k_off, int v_off, int gate_off, const void* z, const void* w2t, const void* w0, int rank, const void* bonus, void* state, long slot_stride,
                            const void* slots, const void* req_indptr, const void* norm, float eps, void* out, int requests, int heads, int dim, int vdim, const void* last_rows, int row_width,
                            long tail_off, int dtype, hipStream_t stream) {
    TL_REQUIRE(requests >= 0 && heads > 0 && ld > 0 && k_off >= 0 && v_off >= 0 && gate_off >= 0 && z && w2t && w0, "wkv_token: bad sizes");
    TL_REQUIRE(tl_wkv_token_fits(rkv, ld, k_off, v_off, gate_off, bonus, state, slot_stride, norm, out, dim, vdim, rank, dtype), "wkv_token: not built for heads of %d x %d or for these places", dim, vdim);
    TL_REQUIRE(slot_stride >= (long)heads * dim * vdim, "wkv_token: the state rows are too short");
    TL_REQUIRE(!last_rows || (row_width > 0 && tail_off >= (long)heads * dim * vdim && slot_stride >= tail_off + row_width),
               "wkv_token: the slots do not hold a row of %d numbers behind the states", row_width);
    TL_REQUIRE(requests <= 65535, "wkv_token: too many requests for one launch");
    if (requests == 0) return TL_OK;
#define TL_WT(T, R, C)                                                                                                                                                          \
    wkv_token_kernel<T, R, C><<<dim3(heads, requests), 256, sizeof(float) * rank, stream>>>((const T*)rkv, ld, k_off, v_off, gate_off, (const float*)z, (const float*)w2t, \
        (const float*)w0, rank, (const float*)bonus, (float*)state, (size_t)slot_stride, (const int*)slots, (const int*)req_indptr, (const float*)norm, eps, (T*)out, heads, dim, vdim, \
        (const float*)last_rows, row_width, (size_t)tail_off)
#define TL_WT_R(T, R) if (vdim <= 64) TL_WT(T, R, 4); else TL_WT(T, R, 8)
#define TL_WT_T(T) if (dim <= 64) { TL_WT_R(T, 4); } else { TL_WT_R(T, 8); }
    if (dtype == TL_DT_F32) { TL_WT_T(float); } else { TL_WT_T(bf16_t); }
#undef TL_WT_T
#undef TL_WT_R
#undef TL_WT
    TL_CHECK_LAUNCH("wkv_token");
    return TL_OK;
}

// ------------------------------------------------------------------ long portions in chunks: recurrences with one decay per head and token
// S <- g S + b k v^T, o = S^T q (the matrix memory; the decayed linear attention) over the tokens of a long portion.
// Token by token the work of a head is a chain that a few compute units walk (four heads of 256 x 512 over 2048 tokens: 1.2 ms, a prompt's
// largest item; in chunks 0.17); cut into chunks of 64 tokens nearly all of it is products of matrices that every chunk can take at once:
//   chunk_states:  D_c = sum_j w_j v_j k_j^T with w_j = b_j prod_{l > j} g_l, and the chunk's decay G_c = prod g;     (all chunks at once)
//   chunk_pass:    S_c, the state before chunk c, from S_0 and the D_c, S_{c+1} = G_c S_c + D_c;                      (a stream over the chunks)
//   chunk_outputs: o_i = G_i S_c^T q_i + sum_{j <= i} b_j (prod_{j < l <= i} g_l) (q_i . k_j) v_j.                     (all chunks at once)
// Products and sums in true 32-bit on v_mfma_f32_32x32x2_f32; decays enter as products of the same numbers the token loop multiplies by (no
// logarithms, no quotients: a decay of zero is one).  Errors against 64 bits are no larger than the token loop's (median per token and head, at 2000 tokens: the matrix memory 1.2e-7 against 1.7e-7, fixed decays 0.70e-7 against 0.79e-7).
// Requests of few tokens in the step (decoded ones) stay with the token loop, which leaves the others out.
#define CK_T 64                 // tokens of a chunk
#define CK_D 64                 // query/key dimensions of a slab in shared memory
#define CK_V 128                // value columns of a work-group
#define CK_LD (CK_D + 4)        // row pitches in shared memory: rows read 16 bytes a lane fall on all banks
#define CK_LV (CK_V + 4)

typedef float ck_f32x16 __attribute__((ext_vector_type(16)));

struct ChunkArgs {
    const void* qkv;            // a token's row: ld numbers; queries of head h from column h * dim on, keys from k_off + h * dim, values from v_off + h * vdim
    int ld, k_off, v_off, heads;
    int dim, vdim;
    const float* gates;         // [tokens][gate_ld]: b at column h * gate_step + b_at, g at h * gate_step + g_at; null: b = 1, g = head_decay[h]
    int gate_ld, gate_step, b_at, g_at;
    const float* head_decay;    // fixed decays
    float qscale, denom_eps;
    float* state;
    size_t slot_stride;
    const int *slots, *req_indptr;
    float* out;                 // [tokens][heads * vdim]
    float *states, *sums, *decays;      // scratch: [chunks][heads][vdim][dim], [chunks][heads][dim] (matrix memory), [chunks][heads]
    int requests, least, seg0, seg_len;      // the tokens seg0 .. seg0 + seg_len - 1 of every request of at least `least` tokens
};

__device__ __forceinline__ int ck_chunks(const ChunkArgs& a, int n) { return n >= a.least && n > a.seg0 ? (min(n - a.seg0, a.seg_len) + CK_T - 1) / CK_T : 0; }

// The request of chunk `want` among all requests' chunks and its first chunk, by a prefix sum over the lanes; -1 beyond the last chunk.
__device__ __forceinline__ int ck_find(const ChunkArgs& a, int want, int& first_chunk) {
    const int lane = threadIdx.x % TL_WAVE;
    int first = 0;
    for (int base = 0; base < a.requests; base += TL_WAVE) {
        const int r = base + lane;
        const int mine = r < a.requests ? ck_chunks(a, a.req_indptr[r + 1] - a.req_indptr[r]) : 0;
        int upto = mine;
#pragma unroll
        for (int o = 1; o < TL_WAVE; o <<= 1) {
            const int t = __shfl_up(upto, o, TL_WAVE);
            if (lane >= o) upto += t;
        }
        const unsigned long long past = __ballot(first + upto > want);
        if (past) {
            const int l = __builtin_amdgcn_readfirstlane(__ffsll(past) - 1);
            first_chunk = first + __builtin_amdgcn_readlane(upto, l) - __builtin_amdgcn_readlane(mine, l);
            return base + l;
        }
        first += __builtin_amdgcn_readlane(upto, TL_WAVE - 1);
    }
    return -1;
}


// MEMORY: the matrix memory (b, g and the running maximum per token; outputs over max(|n . q|, exp(-m)) + denom_eps); otherwise fixed decays.
template <typename T, bool MEMORY>
__global__ void __launch_bounds__(256)
chunk_states_kernel(ChunkArgs a) {
    __shared__ __attribute__((aligned(16))) float sk[CK_T * CK_LD], sv[CK_T * CK_LV];
    __shared__ float sw[CK_T], sn[4 * CK_D];
    const int tid = threadIdx.x, wave = tid / TL_WAVE, lane = tid % TL_WAVE, li = lane & 31, half = lane >> 5;
    int chunk0 = 0;
    const int chunk = blockIdx.x, req = ck_find(a, chunk, chunk0);
    if (req < 0) return;
    const int head = blockIdx.y, v0 = blockIdx.z * CK_V;
    const int tok0 = a.req_indptr[req] + a.seg0 + (chunk - chunk0) * CK_T;
    const int nt = min(min(CK_T, a.req_indptr[req + 1] - tok0), a.seg_len - (chunk - chunk0) * CK_T);
    if (wave == 0) {                                   // the tokens' weights: a product over the tokens behind them, taken from the back
        float b = 0.f, g = 1.f;
        if (lane < nt) {
            if (!MEMORY) { b = 1.f; g = a.head_decay[head]; }
            else {
                const float* row = a.gates + (size_t)(tok0 + lane) * a.gate_ld + head * a.gate_step;
                b = row[a.b_at];
                g = row[a.g_at];
            }
        }
        double p = g;
#pragma unroll
        for (int o = 1; o < TL_WAVE; o <<= 1) {
            const double t = __shfl_down(p, o, TL_WAVE);
            if (lane + o < TL_WAVE) p *= t;
        }
        const double behind = __shfl_down(p, 1, TL_WAVE);
        sw[lane] = (float)(b * (lane + 1 < TL_WAVE ? behind : 1.0));
        if (lane == 0 && blockIdx.z == 0) a.decays[(size_t)chunk * a.heads + head] = (float)p;
    }
    __syncthreads();
    const T* base = (const T*)a.qkv + (size_t)tok0 * a.ld;
    const T* vsrc = base + a.v_off + head * a.vdim + v0;
#pragma unroll
    for (int j = 0; j < CK_T * CK_V / 4 / 256; ++j) {
        const int idx = tid + j * 256, t = idx / (CK_V / 4), c = (idx % (CK_V / 4)) * 4;
        float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
        if (t < nt && v0 + c < a.vdim) {
            x = load4(vsrc + (size_t)t * a.ld + c);
            const float w = sw[t];
            x.x *= w; x.y *= w; x.z *= w; x.w *= w;
        }
        *(float4*)(sv + t * CK_LV + c) = x;
    }
    const T* ksrc = base + a.k_off + head * a.dim;
    float* dst = a.states + ((size_t)chunk * a.heads + head) * a.vdim * a.dim;
    for (int d0 = 0; d0 < a.dim; d0 += CK_D) {
        if (d0 > 0) __syncthreads();
#pragma unroll
        for (int j = 0; j < CK_T * CK_D / 4 / 256; ++j) {
            const int idx = tid + j * 256, t = idx / (CK_D / 4), c = (idx % (CK_D / 4)) * 4;
            *(float4*)(sk + t * CK_LD + c) = t < nt && d0 + c < a.dim ? load4(ksrc + (size_t)t * a.ld + d0 + c) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        __syncthreads();
        if (v0 + wave * 32 < a.vdim) {
            ck_f32x16 acc[2], more[2];                 // two chains of sums each
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[0][i] = acc[1][i] = more[0][i] = more[1][i] = 0.f;
#pragma unroll 4
            for (int t = 0; t < CK_T; t += 4) {
                const float x = sv[(t + half) * CK_LV + wave * 32 + li], y = sv[(t + 2 + half) * CK_LV + wave * 32 + li];
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, sk[(t + half) * CK_LD + li], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, sk[(t + half) * CK_LD + 32 + li], acc[1], 0, 0, 0);
                more[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(y, sk[(t + 2 + half) * CK_LD + li], more[0], 0, 0, 0);
                more[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(y, sk[(t + 2 + half) * CK_LD + 32 + li], more[1], 0, 0, 0);
            }
            acc[0] += more[0];
            acc[1] += more[1];
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int v = v0 + wave * 32 + 8 * (i / 4) + 4 * half + i % 4, d = d0 + 32 * n + li;
                    if (v < a.vdim && d < a.dim) dst[(size_t)v * a.dim + d] = acc[n][i];
                }
        }
        if (MEMORY && blockIdx.z == 0) {            // the keys' own weighted sum (the memory's column of ones)
            const int d = tid % CK_D, part = tid / CK_D;
            float s = 0.f;
#pragma unroll
            for (int t = 0; t < CK_T / 4; ++t) s = fmaf(sw[part * (CK_T / 4) + t], sk[(part * (CK_T / 4) + t) * CK_LD + d], s);
            sn[part * CK_D + d] = s;
            __syncthreads();
            if (tid < CK_D && d0 + tid < a.dim)
                a.sums[((size_t)chunk * a.heads + head) * a.dim + d0 + tid] = ((sn[tid] + sn[CK_D + tid]) + sn[2 * CK_D + tid]) + sn[3 * CK_D + tid];
        }
    }
}

// The states before every chunk, in place of the chunks' own sums, and the state after the last one in the request's slot.  A thread owns four
// neighbouring numbers of a column.  ROWS: the slot holds the state row by row ([dim][vdim], and behind it the keys' sums and the running maximum),
// so a work-group takes a tile of 32 x 32 and turns it in shared memory on its way from and to the slot; otherwise column by column, as the scratch does.
template <bool ROWS>
__global__ void __launch_bounds__(256)
chunk_pass_kernel(ChunkArgs a) {
    __shared__ float turn[32][33];
    const int req = blockIdx.z, head = blockIdx.y, tid = threadIdx.x, lane = tid % TL_WAVE;
    const int count = ck_chunks(a, a.req_indptr[req + 1] - a.req_indptr[req]);
    if (count == 0) return;
    int first = 0;
    for (int base = 0; base < req; base += TL_WAVE) {
        const int r = base + lane;
        int mine = r < req ? ck_chunks(a, a.req_indptr[r + 1] - a.req_indptr[r]) : 0;
#pragma unroll
        for (int o = TL_WAVE / 2; o > 0; o >>= 1) mine += __shfl_xor(mine, o, TL_WAVE);
        first += mine;
    }
    const size_t slot_head = ROWS ? (size_t)a.dim * a.vdim + a.dim + 1 : (size_t)a.dim * a.vdim;
    float* st = a.state + (size_t)a.slots[req] * a.slot_stride + head * slot_head;
    const float* gs = a.decays + (size_t)first * a.heads + head;
    const size_t step = (size_t)a.heads * a.vdim * a.dim;
    const int tiles_d = (a.dim + 31) / 32;
    if (ROWS && (int)blockIdx.x == tiles_d * ((a.vdim + 31) / 32)) {      // the keys' sums and the running maximum
        for (int d = tid; d < a.dim; d += 256) {
            float n = st[(size_t)a.dim * a.vdim + d];
            for (int c = 0; c < count; ++c) {
                float* p = a.sums + ((size_t)(first + c) * a.heads + head) * a.dim + d;
                const float x = *p;
                *p = n;
                n = fmaf(gs[(size_t)c * a.heads], n, x);
            }
            st[(size_t)a.dim * a.vdim + d] = n;
        }
        if (tid == 0) {
            const int end = min(a.req_indptr[req + 1], a.req_indptr[req] + a.seg0 + a.seg_len);
            st[(size_t)a.dim * a.vdim + a.dim] = a.gates[(size_t)(end - 1) * a.gate_ld + head * a.gate_step + 2];
        }
        return;
    }
    int v, d;
    if (ROWS) {
        const int tv = blockIdx.x / tiles_d * 32, td = blockIdx.x % tiles_d * 32;
        v = tv + tid / 8;
        d = td + tid % 8 * 4;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int dd = td + tid / 32 + 8 * j, vv = tv + tid % 32;
            turn[tid / 32 + 8 * j][tid % 32] = dd < a.dim && vv < a.vdim ? st[(size_t)dd * a.vdim + vv] : 0.f;
        }
        __syncthreads();
    } else {
        const int idx = (blockIdx.x * 256 + tid) * 4;
        v = idx / a.dim;
        d = idx % a.dim;
    }
    const bool ok = v < a.vdim && d < a.dim;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    if (ok) {
        if (ROWS) s = make_float4(turn[tid % 8 * 4][tid / 8], turn[tid % 8 * 4 + 1][tid / 8], turn[tid % 8 * 4 + 2][tid / 8], turn[tid % 8 * 4 + 3][tid / 8]);
        else s = *(const float4*)(st + (size_t)v * a.dim + d);
        float* p = a.states + ((size_t)first * a.heads + head) * a.vdim * a.dim + (size_t)v * a.dim + d;
        constexpr int AHEAD = 8;                       // chunks' numbers requested together
        for (int c0 = 0; c0 < count; c0 += AHEAD) {
            float4 x[AHEAD];
            float g[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                const int c = min(c0 + u, count - 1);
                x[u] = *(const float4*)(p + c * step);
                g[u] = gs[(size_t)c * a.heads];
            }
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                if (c0 + u < count) {
                    *(float4*)(p + (c0 + u) * step) = s;
                    s.x = fmaf(g[u], s.x, x[u].x);
                    s.y = fmaf(g[u], s.y, x[u].y);
                    s.z = fmaf(g[u], s.z, x[u].z);
                    s.w = fmaf(g[u], s.w, x[u].w);
                }
            }
        }
        if (!ROWS) *(float4*)(st + (size_t)v * a.dim + d) = s;
    }
    if (ROWS) {
        __syncthreads();
        turn[tid % 8 * 4][tid / 8] = s.x; turn[tid % 8 * 4 + 1][tid / 8] = s.y; turn[tid % 8 * 4 + 2][tid / 8] = s.z; turn[tid % 8 * 4 + 3][tid / 8] = s.w;
        __syncthreads();
        const int tv = blockIdx.x / tiles_d * 32, td = blockIdx.x % tiles_d * 32;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int dd = td + tid / 32 + 8 * j, vv = tv + tid % 32;
            if (dd < a.dim && vv < a.vdim) st[(size_t)dd * a.vdim + vv] = turn[tid / 32 + 8 * j][tid % 32];
        }
    }
}

template <typename T, bool MEMORY>
__global__ void __launch_bounds__(256, 2)
chunk_outputs_kernel(ChunkArgs a) {
    extern __shared__ __attribute__((aligned(16))) float ck_smem[];
    float* sq = ck_smem;                               // [64][CK_LD] queries of a slab; after the slabs the weighted scores
    float* sk = sq + CK_T * CK_LD;                     // [64][CK_LD] keys of a slab
    float* ss = sk + CK_T * CK_LD;                     // [CK_V][CK_LD] the state's columns of a slab; after the slabs [64][CK_LV] values
    float* sg = ss + CK_V * CK_LD;                     // [64] g, [64] b, [64] G (products up to the token), [64] 1 / denominator, [64] keys' sums of a slab
    int* odd = (int*)(sg + 5 * CK_T);                  // whether some value of the chunk is an infinity or a NaN
    const int tid = threadIdx.x, wave = tid / TL_WAVE, lane = tid % TL_WAVE, li = lane & 31, half = lane >> 5;
    int chunk0 = 0;
    const int chunk = blockIdx.x, req = ck_find(a, chunk, chunk0);
    if (req < 0) return;
    const int head = blockIdx.y, v0 = blockIdx.z * CK_V;
    const int tok0 = a.req_indptr[req] + a.seg0 + (chunk - chunk0) * CK_T;
    const int nt = min(min(CK_T, a.req_indptr[req + 1] - tok0), a.seg_len - (chunk - chunk0) * CK_T);
    float m_mine = 0.f;                                // the running maximum after token tid / 4
    if (tid == 0) *odd = 0;
    if (wave == 0) {
        float b = 0.f, g = 1.f;
        if (lane < nt) {
            if (!MEMORY) { b = 1.f; g = a.head_decay[head]; }
            else {
                const float* row = a.gates + (size_t)(tok0 + lane) * a.gate_ld + head * a.gate_step;
                b = row[a.b_at];
                g = row[a.g_at];
            }
        }
        double p = g;
#pragma unroll
        for (int o = 1; o < TL_WAVE; o <<= 1) {
            const double t = __shfl_up(p, o, TL_WAVE);
            if (lane >= o) p *= t;
        }
        sg[lane] = g; sg[CK_T + lane] = b; sg[2 * CK_T + lane] = (float)p;
    }
    if (MEMORY && tid / 4 < nt) m_mine = a.gates[(size_t)(tok0 + tid / 4) * a.gate_ld + head * a.gate_step + 2];
    const T* base = (const T*)a.qkv + (size_t)tok0 * a.ld;
    const T* qsrc = base + head * a.dim;
    const T* ksrc = base + a.k_off + head * a.dim;
    const T* vsrc = base + a.v_off + head * a.vdim + v0;
    const float* src = a.states + ((size_t)chunk * a.heads + head) * a.vdim * a.dim;
    const float* nsrc = a.sums + ((size_t)chunk * a.heads + head) * a.dim;
    const bool cols = v0 + wave * 32 < a.vdim;         // this wave's 32 columns hold some of the head's
    const int ti = wave >> 1, tj = wave & 1;           // this wave's block of the scores
    // sums over 32 dimensions (and below over 32 tokens) in a chain, the chains added up: a single chain over 256 lost more than the token loop's sums
    ck_f32x16 sc, so[2];                               // scores of the wave's block; the state's share of the outputs
#pragma unroll
    for (int i = 0; i < 16; ++i) sc[i] = so[0][i] = so[1][i] = 0.f;
    float qn = 0.f;
    for (int d0 = 0; d0 < a.dim; d0 += CK_D) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < CK_T * CK_D / 4 / 256; ++j) {
            const int idx = tid + j * 256, t = idx / (CK_D / 4), c = (idx % (CK_D / 4)) * 4;
            float4 x = make_float4(0.f, 0.f, 0.f, 0.f), y = x;
            if (t < nt && d0 + c < a.dim) {
                x = load4(qsrc + (size_t)t * a.ld + d0 + c);
                y = load4(ksrc + (size_t)t * a.ld + d0 + c);
                x.x *= a.qscale; x.y *= a.qscale; x.z *= a.qscale; x.w *= a.qscale;
            }
            *(float4*)(sq + t * CK_LD + c) = x;
            *(float4*)(sk + t * CK_LD + c) = y;
        }
#pragma unroll
        for (int j = 0; j < CK_V * CK_D / 4 / 256; ++j) {
            const int idx = tid + j * 256, v = idx / (CK_D / 4), c = (idx % (CK_D / 4)) * 4;
            *(float4*)(ss + v * CK_LD + c) = v0 + v < a.vdim && d0 + c < a.dim ? *(const float4*)(src + (size_t)(v0 + v) * a.dim + d0 + c) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        if (MEMORY && tid < CK_D) sg[4 * CK_T + tid] = d0 + tid < a.dim ? nsrc[d0 + tid] : 0.f;
        __syncthreads();
        if (MEMORY) {
            const float* qr = sq + (tid / 4) * CK_LD + 16 * (tid % 4);
#pragma unroll
            for (int e = 0; e < 16; ++e) qn = fmaf(qr[e], sg[4 * CK_T + 16 * (tid % 4) + e], qn);
        }
        // a lane reads four neighbouring dimensions at once, the two halves of the wave alternate groups of four
        for (int dh = 0; dh < CK_D; dh += 32) {
            ck_f32x16 scx, sox[2];
#pragma unroll
            for (int i = 0; i < 16; ++i) scx[i] = sox[0][i] = sox[1][i] = 0.f;
#pragma unroll
            for (int d = dh; d < dh + 32; d += 8) {
                const float4 q0 = *(const float4*)(sq + li * CK_LD + d + 4 * half), q1 = *(const float4*)(sq + (32 + li) * CK_LD + d + 4 * half);
                const float4 kk = *(const float4*)(sk + (32 * tj + li) * CK_LD + d + 4 * half), sv4 = *(const float4*)(ss + (32 * wave + li) * CK_LD + d + 4 * half);
                const float qa[2][4] = {{q0.x, q0.y, q0.z, q0.w}, {q1.x, q1.y, q1.z, q1.w}}, ka[4] = {kk.x, kk.y, kk.z, kk.w}, va[4] = {sv4.x, sv4.y, sv4.z, sv4.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (tj <= ti) scx = __builtin_amdgcn_mfma_f32_32x32x2f32(ti ? qa[1][e] : qa[0][e], ka[e], scx, 0, 0, 0);
                    if (cols) {
                        sox[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(qa[0][e], va[e], sox[0], 0, 0, 0);
                        sox[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(qa[1][e], va[e], sox[1], 0, 0, 0);
                    }
                }
            }
            sc += scx;
            so[0] += sox[0];
            so[1] += sox[1];
        }
    }
    __syncthreads();
    // the weights b_j prod_{j < l <= i} g_l of every pair of tokens, lane j's column row after row (each wave the rows of its quarter), and the values
    {
        double r = 0.0;
        const double bj = sg[CK_T + lane];
        const int end = 16 * wave + 16;
#pragma unroll 4
        for (int i = 0; i < end; ++i) {
            r = i == lane ? bj : r * sg[i];
            if (i >= end - 16) sq[i * CK_LD + lane] = i < lane ? 0.f : (float)r;
        }
    }
#pragma unroll
    for (int j = 0; j < CK_T * CK_V / 4 / 256; ++j) {
        const int idx = tid + j * 256, t = idx / (CK_V / 4), c = (idx % (CK_V / 4)) * 4;
        const float4 x = t < nt && v0 + c < a.vdim ? load4(vsrc + (size_t)t * a.ld + c) : make_float4(0.f, 0.f, 0.f, 0.f);
        *(float4*)(ss + t * CK_LV + c) = x;
        if (fmaf(x.x, 0.f, fmaf(x.y, 0.f, fmaf(x.z, 0.f, x.w * 0.f))) != 0.f) *odd = 1;      // an infinity or a NaN
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {                     // (a score of a later token, which may be anything, is put aside and not multiplied by zero)
        const int row = 32 * ti + 8 * (i / 4) + 4 * half + i % 4, col = 32 * tj + li;
        float* w = sq + row * CK_LD + col;
        if (tj <= ti && col <= row) *w *= sc[i];
    }
    ck_f32x16 o[2], o1;                                // the chunk's own share, apart from the state's: of its first 32 tokens, of its last
#pragma unroll
    for (int i = 0; i < 16; ++i) o[0][i] = o[1][i] = o1[i] = 0.f;
    __syncthreads();
    if (MEMORY) {
        // n . q after every token: the state's share and the chunk's, four lanes a token
        const float* w = sq + (tid / 4) * CK_LD + 16 * (tid % 4);
        float rs = 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e) rs += w[e];
        float den = fmaf(sg[2 * CK_T + tid / 4], qn, rs);
        den += row_exchange<0xB1>(den);
        den += row_exchange<0x4E>(den);
        if (tid % 4 == 0) sg[3 * CK_T + tid / 4] = fmaxf(fabsf(den), expf(-m_mine)) + a.denom_eps;
        __syncthreads();
    }
    if (!cols) return;
    if (*odd) {
        // some value is an infinity or a NaN: the matrix products would carry it, times a weight of zero, to the tokens before it as well
        for (int t = 0; t < nt; ++t) {
            const float x = ss[t * CK_LV + wave * 32 + li];
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int row = 32 * n + 8 * (i / 4) + 4 * half + i % 4;
                    if (row >= t) o[n][i] = fmaf(sq[row * CK_LD + t], x, o[n][i]);
                }
        }
    } else {
#pragma unroll 4
        for (int t = 0; t < CK_T; t += 8) {
            const float4 w1 = *(const float4*)(sq + (32 + li) * CK_LD + t + 4 * half);
            const float wa[4] = {w1.x, w1.y, w1.z, w1.w};
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = ss[(t + 4 * half + e) * CK_LV + wave * 32 + li];
            if (t < 32) {                                  // (the first 32 tokens see none of the last 32)
                const float4 w0 = *(const float4*)(sq + li * CK_LD + t + 4 * half);
                const float wb[4] = {w0.x, w0.y, w0.z, w0.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    o[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(wb[e], x[e], o[0], 0, 0, 0);
                    o[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(wa[e], x[e], o[1], 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) o1 = __builtin_amdgcn_mfma_f32_32x32x2f32(wa[e], x[e], o1, 0, 0, 0);
            }
        }
        o[1] += o1;
    }
    const int v = v0 + wave * 32 + li;
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int row = 32 * n + 8 * (i / 4) + 4 * half + i % 4;
            if (row >= nt || v >= a.vdim) continue;
            float y = fmaf(sg[2 * CK_T + row], so[n][i], o[n][i]);
            if (MEMORY) y /= sg[3 * CK_T + row];
            a.out[((size_t)(tok0 + row) * a.heads + head) * a.vdim + v] = y;
        }
}

// How the long portions of a step go through the chunks: `segment` tokens of every portion a pass, `grid` chunks of them all in a pass at most, whose
// states and sums stand in `scratch` (`floats` numbers).
struct ChunkPlan {
    int segment, grid;
    float* scratch;
    long floats;
};

template <typename T, bool MEMORY>
static int launch_chunks(ChunkArgs a, const ChunkPlan& p, int longest, hipStream_t stream) {
    const size_t per_chunk = (size_t)a.heads * ((size_t)a.vdim * a.dim + (MEMORY ? a.dim : 0) + 1);
    TL_REQUIRE(p.segment > 0 && p.segment % CK_T == 0 && p.grid > 0 && p.floats >= (long)(p.grid * per_chunk), "chunked scan: scratch of %ld numbers does not hold %d chunks", p.floats, p.grid);
    const int chunks = p.grid;
    float* scratch = p.scratch;
    a.seg_len = p.segment;
    a.states = scratch;
    a.sums = scratch + (size_t)chunks * a.heads * a.vdim * a.dim;
    a.decays = a.sums + (MEMORY ? (size_t)chunks * a.heads * a.dim : 0);
    constexpr size_t smem = sizeof(float) * (2 * CK_T * CK_LD + CK_V * CK_LD + 5 * CK_T + 4);
    auto outputs = chunk_outputs_kernel<T, MEMORY>;
    static hipError_t allowed = hipFuncSetAttribute((const void*)outputs, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    if (allowed != hipSuccess) { tl_set_error("chunked scan: cannot get %zu bytes of shared memory: %s", smem, hipGetErrorString(allowed)); return TL_ERR_HIP; }
    const dim3 grid(chunks, a.heads, (a.vdim + CK_V - 1) / CK_V);
    const dim3 pass(MEMORY ? (a.dim + 31) / 32 * ((a.vdim + 31) / 32) + 1 : (a.vdim * a.dim / 4 + 255) / 256, a.heads, a.requests);
    for (a.seg0 = 0; a.seg0 < longest; a.seg0 += a.seg_len) {
        chunk_states_kernel<T, MEMORY><<<grid, 256, 0, stream>>>(a);
        TL_CHECK_LAUNCH("chunk_states");
        chunk_pass_kernel<MEMORY><<<pass, 256, 0, stream>>>(a);
        TL_CHECK_LAUNCH("chunk_pass");
        outputs<<<grid, 256, smem, stream>>>(a);
        TL_CHECK_LAUNCH("chunk_outputs");
    }
    return TL_OK;
}

// What the matrix memory's chunks read: per token and head (decay, input factor, running maximum, 0), the maximum taken from the slot's on as a
// scan over 64 tokens at a time (max-plus: a stretch is the pair (sum of the log forget gates, maximum it brings)).  A work-group a request and head, a stretch of 64 to
// each of its up to sixteen waves, which meet once a round: what a round costs is a trip to memory and the scan within a wave, 1.1 us, and one wave alone
// went through 31 rounds of them for 2000 tokens (35.5 us; now 9.5).  A wave takes the stretches before its own in their order, so the sums are one wave's.
#define MG_WAVES 16
__global__ void __launch_bounds__(MG_WAVES * TL_WAVE)
mlstm_gates_kernel(const float* __restrict__ gates, const float* __restrict__ state, size_t slot_stride, const int* __restrict__ slots,
                   const int* __restrict__ req_indptr, float4* __restrict__ factors, int heads, int dim, int vdim, float cap, int least) {
    __shared__ float2 stretch[2][MG_WAVES];
    const int req = blockIdx.y, head = blockIdx.x, lane = threadIdx.x % TL_WAVE, wave = threadIdx.x / TL_WAVE, waves = blockDim.x / TL_WAVE;
    const int tok0 = req_indptr[req], tok1 = req_indptr[req + 1];
    if (tok1 - tok0 < least) return;
    float m = state[(size_t)slots[req] * slot_stride + (size_t)(head + 1) * ((size_t)dim * vdim + dim + 1) - 1];
    for (int base = tok0, round = 0; base < tok1; base += blockDim.x, round ^= 1) {
        const int t = base + threadIdx.x;
        const float* g = gates + (size_t)min(t, tok1 - 1) * 2 * heads;
        const float gi = soft_cap(g[head], cap), gf = log_sigmoid(soft_cap(g[heads + head], cap));
        float f = gf, i = gi;                          // of the stretch that ends with this lane's token
#pragma unroll
        for (int o = 1; o < TL_WAVE; o <<= 1) {
            const float pf = __shfl_up(f, o, TL_WAVE), pi = __shfl_up(i, o, TL_WAVE);
            if (lane >= o) { i = fmaxf(pi + f, i); f += pf; }
        }
        if (lane == TL_WAVE - 1) stretch[round][wave] = make_float2(f, i);
        __syncthreads();                               // (two sets in turn: the next round's are written while the slowest wave still reads these)
        float at = m;                                  // the maximum as this wave's stretch finds it, and m as the next round does
        for (int w = 0; w < waves; ++w) {
            if (w == wave) at = m;
            const float2 all = stretch[round][w];
            m = fmaxf(all.x + m, all.y);
        }
        const float mine = fmaxf(f + at, i);
        float before = __shfl_up(mine, 1, TL_WAVE);
        if (lane == 0) before = at;
        if (t < tok1) factors[(size_t)t * heads + head] = make_float4(expf(gf + before - mine), expf(gi - mine), mine, 0.f);
    }
}

// Whether a step's long portions (count of them, tokens in all, `chunks` chunks in `passes` passes, the longest of so many tokens) go through the chunks, beside
// `rest` requests of rest_tokens tokens, rest_longest at most: two estimates in us, fitted to the device's times below.
//   The token loop.  Fixed decays: a token of the longest portion 0.18 (0.115 with states of 64 rows), or all portions' work-groups over 2.8 of them a compute
//     unit, and behind it the others' over 2.4, whose one token is a batch of 16 like any.  The matrix memory: a token 0.58, 1.2 or 2.8 by the rows a lane keeps, once for
//     every round of work-groups (16 waves a compute unit); the decoded requests' states cost the same on both ways.
//   The chunks: their launches, a little for every chunk of the longest portion, the chunks' sums and products; then the others go through the loop alone, decoded ones in
//     batches of one token.
// Measured (us, loop / chunks): fixed decays, 16 heads of 128 x 128: 128 tokens 24 / 45, 256 51 / 47, 2048 367 / 80; 16 x 128 78 / 83; 64 beside 31 decoded 38 / 65, 128 beside
// 31 47 / 66, 512 beside 31 114 / 70, 256 beside 200 158 / 133; 32 heads: 256 51 / 52, 256 beside 31 93 / 79; 4 heads of 64 x 64: 256 32 / 32, beside 8 32 / 35.  The matrix memory, 4
// heads of 256 x 512: 64 tokens 49 / 77, 128 85 / 79, 2048 1191 / 170; 32 beside 8 decoded 127 / 122, 64 beside 31 278 / 194, 32 beside 63 269 / 269, 32 beside 8 of 20 176 / 220, 128 beside them
// 445 / 229; 8 heads: 64 91 / 80, 32 beside 63 521 / 541; 2 heads of 128 x 128: 64 44 / 52, 128 80 / 54, 64 beside 31 57 / 76, 64 beside 63 103 / 84, 16 x 64 52 / 56.
extern "C" int tl_chunks_pay(int memory, int count, int tokens, int chunks, int passes, int longest, int rest, int rest_tokens, int rest_longest, int requests, int heads,
                             int dim, int vdim) {
    const double state = (double)heads * dim * vdim;
    if (rest_tokens == 0) rest = rest_longest = 0;                 // (none, or the caller cannot tell)
    if (memory) {
        const MlstmShape shape = mlstm_shape(requests, heads, dim, vdim);
        const int waves = (dim + shape.rpt * (TL_WAVE / shape.cols) - 1) / (shape.rpt * (TL_WAVE / shape.cols));
        const double token = shape.rpt <= 4 ? 0.58 : shape.rpt <= 8 ? 1.2 : 0.175 * shape.rpt, tiles = (double)heads * ((vdim + shape.cols - 2) / (shape.cols - 1));
        const double at_once = (double)tl_mlstm_units * (waves < 16 ? 16 / waves : 1);
        auto loop = [&](int n, int most) { return n > 0 && most > 1 ? most * token * ceil(n * tiles / at_once) : 0.0; };
        const double others = loop(rest, rest_longest), together = loop(count + (rest_longest > 1 ? rest : 0), longest > rest_longest ? longest : rest_longest);
        const double all = fmin(loop(count, longest) + others, together) + (rest > 0 ? 0 : 10);
        return 50 + 25 * fmin(1.0, state / 5e5) + longest * 0.02 + chunks * 64 * state * 5e-8 + (passes - 1) * 50.0 + (rest > 0 ? 15 + others : 0) < all;
    }
    const double groups = (double)((vdim + DELTA_COLS - 1) / DELTA_COLS) * heads, token = dim <= 64 ? 0.115 : 0.18;
    auto batches = [&](int n, int t, double per_unit) { return token * groups * (t + (DELTA_TB - 1.0) * n) / (per_unit * tl_mlstm_units); };
    const double all = 3 + fmax(token * longest, batches(count, tokens, 2.8)) + batches(rest, rest_tokens, 2.4);
    const double others = rest == 0 ? 0 : 5 + (rest_longest <= 1 ? 1.4e-6 * rest * state : batches(rest, rest_tokens, 2.4));
    return 30 + 12 * fmin(1.0, state / 262144) + longest * 0.003 + chunks * 64 * state * 1e-7 + (passes - 1) * 30.0 + others < all;
}

// Whether the chunks can be read in whole pieces of four numbers.
static bool chunks_fit(const void* qkv, int ld, int k_off, int v_off, int dim, int vdim, const void* state, long slot_stride, bool columns) {
    return dim % 4 == 0 && vdim % 4 == 0 && ld % 4 == 0 && k_off % 4 == 0 && v_off % 4 == 0 && ((uintptr_t)qkv & 15) == 0 &&
           (!columns || (((uintptr_t)state & 15) == 0 && slot_stride % 4 == 0));
}

// qkv [tokens, ld]: queries at column 0 (heads * dim), keys at k_off, values at v_off (heads * vdim); gates float
// [tokens, 2 * heads]; state float [slots, heads, dim * vdim + dim + 1] with slot_stride floats between slots;
// out float [tokens, heads * vdim]; before: scratch of requests * heads * (dim + 1) floats.  Requests whose req_indptr range
// is empty are left alone.  longest: no fewer tokens than any request of the step brings.  With scratch (null: the token loop alone) requests of at least `least`
// tokens go through the chunks where the rows allow it: `segment` tokens of each a pass, chunk_grid chunks a pass at most; the chunks' states come first in
// scratch and from scratch_floats on the tokens' factors (4 * tokens * heads floats).  The token loop then takes the others (rest: how many there are, or more if
// the caller cannot tell; 0 only if there are none), of about rest_longest tokens at most, which sizes its batches.
extern "C" int tl_mlstm_scan(const void* qkv, int ld, int k_off, int v_off, const void* gates, void* state, long slot_stride,
                             const void* slots, const void* before, const void* req_indptr, void* out, int requests, int heads, int dim, int vdim,
                             float cap, float qscale, float denom_eps, int longest, int segment, int chunk_grid, int least, int rest, int rest_longest,
                             void* scratch, long scratch_floats, int dtype, hipStream_t stream) {
    TL_REQUIRE(requests >= 0 && heads > 0 && dim > 0 && vdim > 0 && ld > 0, "mlstm_scan: bad sizes");
    TL_REQUIRE(dim <= 1024, "mlstm_scan: built for up to 1024 query/key dimensions per head, got %d", dim);
    TL_REQUIRE(slot_stride >= (long)heads * ((long)dim * vdim + dim + 1), "mlstm_scan: the state rows are too short");
    TL_REQUIRE(dtype == TL_DT_F32 || dtype == TL_DT_BF16, "mlstm_scan: unknown dtype %d", dtype);
    if (requests == 0) return TL_OK;
    const bool chunks = scratch && longest >= least && chunks_fit(qkv, ld, k_off, v_off, dim, vdim, state, slot_stride, false);
    if (chunks) {
        float4* factors = (float4*)((float*)scratch + scratch_floats);
        mlstm_gates_kernel<<<dim3(heads, requests), TL_WAVE * max(1, min(MG_WAVES, (longest + TL_WAVE - 1) / TL_WAVE)), 0, stream>>>((const float*)gates, (const float*)state, (size_t)slot_stride, (const int*)slots,
                                                                     (const int*)req_indptr, factors, heads, dim, vdim, cap, least);
        TL_CHECK_LAUNCH("mlstm_gates");
        const ChunkArgs a{qkv, ld, k_off, v_off, heads, dim, vdim, (const float*)factors, 4 * heads, 4, 1, 0, nullptr, qscale, denom_eps, (float*)state,
                          (size_t)slot_stride, (const int*)slots, (const int*)req_indptr, (float*)out, nullptr, nullptr, nullptr, requests, least, 0, 0};
        const ChunkPlan plan{segment, chunk_grid, (float*)scratch, scratch_floats};
        const int rc = dtype == TL_DT_F32 ? launch_chunks<float, true>(a, plan, longest, stream) : launch_chunks<bf16_t, true>(a, plan, longest, stream);
        if (rc != TL_OK || rest == 0) return rc;
    }
    return mlstm_token_loop(qkv, ld, k_off, v_off, gates, state, slot_stride, slots, before, req_indptr, out, requests, heads, dim, vdim, cap, qscale, denom_eps,
                            chunks ? rest_longest : longest, chunks ? least : INT_MAX, dtype, stream);
}

// ------------------------------------------------------------------ decayed linear attention
// Per head S <- decay[head] S + k v^T, o = S^T q over the step's tokens, request by request from the state its slot holds: qkv float
// [T, 2 * heads * dim + heads * vdim] (queries, keys, values, head by head), state as the delta rule's, out float [T, heads * vdim].
extern "C" int tl_decay_scan(const void* qkv, const void* decay, void* state, long slot_stride, const void* slots, const void* req_indptr,
                             void* out, int requests, int heads, int dim, int vdim, int tokens, int longest, int segment, int chunk_grid, int least, int rest,
                             int rest_longest, void* scratch, long scratch_floats, hipStream_t stream) {
    TL_REQUIRE(requests >= 0 && heads > 0 && dim > 0 && vdim > 0 && decay, "decay_scan: bad sizes");
    TL_REQUIRE(dim <= DELTA_L * 16, "decay_scan: built for up to %d query/key dimensions per head, got %d", DELTA_L * 16, dim);
    TL_REQUIRE(slot_stride >= (long)heads * dim * vdim, "decay_scan: the state rows are too short");
    TL_REQUIRE(requests <= 65535 && heads <= 65535, "decay_scan: too many requests or heads for one launch");
    if (requests == 0) return TL_OK;
    const bool chunks = scratch && longest >= least && chunks_fit(qkv, 2 * heads * dim + heads * vdim, 0, 0, dim, vdim, state, slot_stride, true);
    if (chunks) {
        const int rc = launch_chunks<float, false>(ChunkArgs{qkv, 2 * heads * dim + heads * vdim, heads * dim, 2 * heads * dim, heads, dim, vdim, nullptr, 0, 0, 0, 0,
            (const float*)decay, 1.f, 0.f, (float*)state, (size_t)slot_stride, (const int*)slots, (const int*)req_indptr, (float*)out, nullptr, nullptr, nullptr,
            requests, least, 0, 0}, ChunkPlan{segment, chunk_grid, (float*)scratch, scratch_floats}, longest, stream);
        if (rc != TL_OK || rest == 0) return rc;
    }
    launch_delta_scan<0>(qkv, nullptr, decay, state, slot_stride, slots, req_indptr, out, requests, heads, heads, dim, vdim, chunks ? rest * rest_longest : tokens,
                         chunks ? rest_longest : longest, chunks ? least : INT_MAX, stream);
    TL_CHECK_LAUNCH("decay_scan");
    return TL_OK;
}

// ------------------------------------------------------------------ selective state-space recurrence (Mamba-2)
// Per head S <- decay S + dt B x^T (S: state x vdim), y = S^T C + D x, with B and C shared by the heads of a group.  qkv float [T, 2 * groups *
// state + heads * vdim] as selective_prepare leaves it (C, B, x), gates float [T, 2 * heads] (dt, decay), skip float [heads] (D); the
// state as the delta rule's ([vdim][state] per head), out float [T, heads * vdim].
extern "C" int tl_selective_scan(const void* qkv, const void* gates, const void* skip, void* state, long slot_stride, const void* slots,
                                 const void* req_indptr, void* out, int requests, int heads, int groups, int dim, int vdim, int tokens, int longest, int least, int blocks,
                                 int rest, int rest_longest, void* scratch, long scratch_floats, hipStream_t stream) {
    TL_REQUIRE(requests >= 0 && heads > 0 && groups > 0 && heads % groups == 0 && dim > 0 && vdim > 0 && gates && skip, "selective_scan: bad sizes");
    TL_REQUIRE(dim <= DELTA_L * 16, "selective_scan: built for states of up to %d numbers per column, got %d", DELTA_L * 16, dim);
    TL_REQUIRE(slot_stride >= (long)heads * dim * vdim, "selective_scan: the state rows are too short");
    TL_REQUIRE(requests <= 65535 && heads <= 65535, "selective_scan: too many requests or heads for one launch");
    if (requests == 0) return TL_OK;
    const bool through = blocks_fit(2, qkv, heads, groups, dim, vdim, state, slot_stride, blocks, scratch, scratch_floats);
    if (through) {
        launch_blocks<2>(qkv, gates, skip, state, slot_stride, slots, req_indptr, out, requests, heads, groups, dim, vdim, least, blocks, scratch, stream);
        TL_CHECK_LAUNCH("selective_blocks");
        if (rest == 0) return TL_OK;
    }
    launch_delta_scan<2>(qkv, gates, skip, state, slot_stride, slots, req_indptr, out, requests, heads, groups, dim, vdim, through ? rest * rest_longest : tokens,
                         through ? rest_longest : longest, through ? least : INT_MAX, stream);
    TL_CHECK_LAUNCH("selective_scan");
    return TL_OK;
}
