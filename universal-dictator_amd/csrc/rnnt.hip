// RNN-T joint and greedy decoding, batched over streams (include/ud_rnnt.h).
//
// The reference decodes one stream at a time on the CPU (Sources/DictatorCore/Decoding/RNNT.swift):
// per emitted token one prediction step (embedding, 2 LSTM layers of [4H, 2H] sgemv, joint.pred)
// and per (frame, symbol) one joint evaluation ([V, H] sgemv).  Here one greedy iteration does
// that work for every active stream of the call at once, as fp32 products over M = active streams
// (the weights are read once per iteration, not once per stream), in four launches:
//
//   predict (streams without a cached prediction):
//     rnnt_lstm_kernel, per layer: gates of [x ; h] . [W_ih | W_hh]^T and the cell: x is the embedding
//                of the last token, then the layer below's new h
//     rnnt_linear_kernel: g = joint.pred of the top h -> the slot's cached g
//   joint (every remaining frame of every active stream, under its current prediction):
//     rnnt_joint_kernel: relu(f_t + g) . W_out^T and the first index of each row's maximum, into mapped
//                host memory
//
// Each of them owns whole K ranges (the 8 waves of a workgroup split K and are summed in LDS), so the
// cell, the sum f + g and the argmax happen where the product ends, and no slab or activation row goes
// through memory between launches.  An iteration is a chain of short kernels that the host waits for:
// with the products split over workgroups it took nine (embedding, a product and a cell per layer, a
// product, the joint's input, a product, the argmax) of 4-8 us each.
// Now, up to 16 rows, 6.0 us per LSTM layer (13 MB of weights, 2.2 TB/s), 3.3 joint.pred, 6.6 the joint.
// More rows cost more, since each of a product's workgroups (160 for a layer, 65 for the joint) reads all of
// them: in a trace 6.3 us a layer up to 16 rows, 10.8 up to 32, 18.4 at 33-64 (0.7 TB/s of weights);
// joint.pred 3.8, 5.2, 9.3; the joint 7.0, 9.5, 14.7.
// A chunk of 2 frames that ends after 10 tokens: one stream 738 -> 373 us, 64 streams 911 -> 472;
// 64 x 14 frames 1,826 -> 1,173.  joint.enc (rnnt_linear_kernel, one launch instead of slabs and their
// sum): 128 rows 17.2 -> 12.2 us.
//
// A slot has two states (h, c of every layer): the committed one and the one its cached prediction
// leaves.  Emitting a token makes the second the first: the host flips the slot's index
// (RNNT.swift:144-147), and nothing is copied.
//
// The host keeps the greedy control (RNNT.swift:125-151): blank ends a frame, at most
// max_symbols tokens per frame, and the prediction for the last token is cached until a token is
// emitted (so frames that end in blank do not rerun the LSTM).  Because a blank leaves the
// prediction unchanged, the joint results of the frames after a blank are known in advance: one
// iteration evaluates them all and the host consumes them up to the first emission.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/ud_rnnt.h"
#include "kernels.hpp"
#include "ud_common.hpp"

int ud_set_error(int code, const char* msg);   // encoder.hip

namespace ud {

constexpr int RNNT_WK = 8;          // waves of a workgroup: the K split of every product

__device__ __forceinline__ float sigmoid_f(float x) { return 1.0f / (1.0f + expf(-x)); }

// Four floats at any 4-byte address (a caller's rows need no more than a float's alignment).
typedef float f32x4u_t __attribute__((ext_vector_type(4), aligned(4)));

// acc[j][i] (transposed 16 x 16 tiles: column tile j, row tile i) += rows . W^T over the 16-wide K
// blocks wave, wave + 8, .. of nkb, on v_mfma_f32_16x16x4_f32.  W: the lane's first column tile in the
// fragment-major layout (frag_index_f32), rows_at(i, kb): the lane's four values of row tile i in K
// block kb.  A row's sum runs in the same order whatever MT and NT are, so its result does not depend
// on the batch it is computed in.
template <int MT, int NT, typename RowsAt>
__device__ __forceinline__ void rows_product(const float* W, int nkb, int wave, RowsAt rows_at, f32x4_t (&acc)[NT][MT]) {
    constexpr int U = MT * NT == 1 ? 4 : MT * NT <= 4 ? 2 : 1;       // K blocks in flight behind U being multiplied
    struct Frags {
        f32x4_t a[MT], b[NT];
    };
    Frags f0[U], f1[U];
    auto load = [&](Frags (&f)[U], int i0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int kb = wave + RNNT_WK * (i0 + u);
            if (kb < nkb) {
#pragma unroll
                for (int j = 0; j < NT; j++) f[u].b[j] = *reinterpret_cast<const f32x4_t*>(W + ((int64_t)j * nkb + kb) * 256);
#pragma unroll
                for (int i = 0; i < MT; i++) f[u].a[i] = rows_at(i, kb);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto mma = [&](const Frags (&f)[U], int i0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; u++)
            if (wave + RNNT_WK * (i0 + u) < nkb) {
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int j = 0; j < NT; j++)
#pragma unroll
                        for (int i = 0; i < MT; i++)
                            acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[u].b[j][e], f[u].a[i][e], acc[j][i], 0, 0, 0);
            }
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++) acc[j][i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    load(f0, 0);
    for (int i0 = 0; wave + RNNT_WK * i0 < nkb; i0 += 2 * U) {
        load(f1, i0 + U);
        mma(f0, i0);
        load(f0, i0 + 2 * U);
        mma(f1, i0 + U);
    }
}

// The workgroup's tile t = j MT + i, summed over its waves in wave order: the lane's row is r16 =
// lane % 16 of row tile i, its columns 4 (lane / 16) .. + 3 of column tile j.
template <int MT, int NT>
__device__ __forceinline__ f32x4_t sum_waves(const f32x4_t (*red)[NT * MT][64], int t, int lane) {
    f32x4_t v = red[0][t][lane];
#pragma unroll
    for (int w = 1; w < RNNT_WK; w++) v += red[w][t][lane];
    return v;
}
template <int MT, int NT>
__device__ __forceinline__ void post_tiles(f32x4_t (*red)[NT * MT][64], const f32x4_t (&acc)[NT][MT], int wave, int lane) {
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++) red[wave][j * MT + i][lane] = acc[j][i];
    __syncthreads();
}

// One LSTM layer for the n listed slots.  W [4H][2H] = [W_ih | W_hh] with the rows of unit j's gates
// i, f, g, o together (rows 4j .. 4j + 3): a 16-column tile holds 4 units, so the lane that ends with
// columns 4q .. 4q + 3 has one unit's four gates and computes its cell.  state: h, then c, of both
// states of every slot and layer, [2][S][L][H] each (StateAt).
struct StateAt {
    float* h;
    float* c;
    int64_t flip;                   // elements between a slot's two states
    int L, H;
};
template <int MT>
__global__ __launch_bounds__(64 * RNNT_WK) void rnnt_lstm_kernel(const float* __restrict__ W, const float* __restrict__ bias,
                                                                 const float* __restrict__ embed, const int32_t* __restrict__ slot,
                                                                 const int32_t* __restrict__ tok, const int32_t* __restrict__ flip,
                                                                 StateAt st, int n, int layer, int blank) {
    __shared__ f32x4_t red[RNNT_WK][MT][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, q = lane >> 4, H = st.H, hb = H / 16, nkb = 2 * hb;
    // the lane's rows: x (null: the blank's embedding, NeMo's zero padding row), then h
    const float *px[MT], *ph[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int b = min((int)(blockIdx.y * MT + i) * 16 + r16, n - 1), s = slot[b], f = flip[b];
        const int64_t so = ((int64_t)s * st.L + layer) * H;
        ph[i] = st.h + f * st.flip + so + 4 * q;
        if (layer > 0) px[i] = st.h + (1 - f) * st.flip + so - H + 4 * q;
        else px[i] = tok[b] == blank ? nullptr : embed + (int64_t)tok[b] * H + 4 * q;
    }
    f32x4_t acc[1][MT];
    rows_product<MT, 1>(W + ((int64_t)blockIdx.x * nkb * 64 + lane) * 4, nkb, wave, [&](int i, int kb) __attribute__((always_inline)) {
        if (kb >= hb) return *reinterpret_cast<const f32x4_t*>(ph[i] + (kb - hb) * 16);
        return px[i] ? *reinterpret_cast<const f32x4_t*>(px[i] + kb * 16) : f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }, acc);
    post_tiles<MT, 1>(red, acc, wave, lane);
    for (int i = wave; i < MT; i += RNNT_WK) {
        const int b = (blockIdx.y * MT + i) * 16 + r16;
        if (b >= n) continue;
        const int j = blockIdx.x * 4 + q;
        const f32x4_t v = sum_waves<MT, 1>(red, i, lane);
        const float ig = sigmoid_f(bias[j] + v[0]), fg = sigmoid_f(bias[H + j] + v[1]);
        const float gg = tanhf(bias[2 * H + j] + v[2]), og = sigmoid_f(bias[3 * H + j] + v[3]);
        const int64_t o = ((int64_t)slot[b] * st.L + layer) * H + j;
        const float cn = fg * st.c[flip[b] * st.flip + o] + ig * gg;
        st.c[(1 - flip[b]) * st.flip + o] = cn;
        st.h[(1 - flip[b]) * st.flip + o] = og * tanhf(cn);
    }
}

// out = rows . W^T + bias: joint.enc over a caller's rows (slot null: row b at x + b K, out row b), or
// joint.pred over the slots' new top h (row at x + (1 - flip) st.flip + (slot L + L - 1) H, out row slot).
template <int MT, int NT>
__global__ __launch_bounds__(64 * RNNT_WK) void rnnt_linear_kernel(const float* __restrict__ W, const float* __restrict__ bias,
                                                                   const float* __restrict__ x, const int32_t* __restrict__ slot,
                                                                   const int32_t* __restrict__ flip, StateAt st,
                                                                   float* __restrict__ out, int n, int N, int K) {
    __shared__ f32x4_t red[RNNT_WK][NT * MT][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, q = lane >> 4, nkb = K / 16;
    const float* px[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int b = min((int)(blockIdx.y * MT + i) * 16 + r16, n - 1);
        const int64_t o = slot ? (1 - flip[b]) * st.flip + ((int64_t)slot[b] * st.L + st.L - 1) * st.H : (int64_t)b * K;
        px[i] = x + o + 4 * q;
    }
    f32x4_t acc[NT][MT];
    rows_product<MT, NT>(W + ((int64_t)blockIdx.x * NT * nkb * 64 + lane) * 4, nkb, wave, [&](int i, int kb) __attribute__((always_inline)) {
        return *reinterpret_cast<const f32x4_t*>(px[i] + kb * 16);
    }, acc);
    post_tiles<MT, NT>(red, acc, wave, lane);
    for (int t = wave; t < NT * MT; t += RNNT_WK) {
        const int b = (blockIdx.y * MT + t % MT) * 16 + r16, c = (blockIdx.x * NT + t / MT) * 16 + 4 * q;
        if (b >= n) continue;
        const f32x4_t v = sum_waves<MT, NT>(red, t, lane) + *reinterpret_cast<const f32x4_t*>(bias + c);
        *reinterpret_cast<f32x4u_t*>(out + (int64_t)(slot ? slot[b] : b) * N + c) = v;
    }
}

// A float's bits ordered as unsigned integers (-0 as +0); 0 is below every float but NaN.
__device__ __forceinline__ uint32_t ordered_bits(float x) {
    const uint32_t u = __float_as_uint(x + 0.0f);
    return u ^ ((u >> 31) ? 0xffffffffu : 0x80000000u);
}

// best[b] = the first index of the maximum of bias + relu(f[erow b] + g[slot b]) . W^T over the V
// columns; -1 if no logit exceeds -inf (NaN logits do not count).  A row's columns lie in many
// workgroups: each posts its maximum as (ordered logit, ~index) with a 64-bit atomic max, whose result
// does not depend on their order, and the last one to finish hands all rows to the host and clears the
// keys and the count for the next launch.
template <int MT, int NT>
__global__ __launch_bounds__(64 * RNNT_WK) void rnnt_joint_kernel(const float* __restrict__ W, const float* __restrict__ bias,
                                                                  const float* __restrict__ f, const float* __restrict__ g,
                                                                  const int32_t* __restrict__ slot, const int32_t* __restrict__ erow,
                                                                  unsigned long long* key, unsigned int* done,
                                                                  int32_t* __restrict__ best, int n, int V, int H) {
    __shared__ f32x4_t red[RNNT_WK][NT * MT][64];
    __shared__ bool is_last;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, q = lane >> 4, nkb = H / 16;
    const float *pf[MT], *pg[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int b = min((int)(blockIdx.y * MT + i) * 16 + r16, n - 1);
        pf[i] = f + (int64_t)erow[b] * H + 4 * q;
        pg[i] = g + (int64_t)slot[b] * H + 4 * q;
    }
    f32x4_t acc[NT][MT];
    rows_product<MT, NT>(W + ((int64_t)blockIdx.x * NT * nkb * 64 + lane) * 4, nkb, wave, [&](int i, int kb) __attribute__((always_inline)) {
        f32x4_t v = *reinterpret_cast<const f32x4u_t*>(pf[i] + kb * 16) + *reinterpret_cast<const f32x4_t*>(pg[i] + kb * 16);
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = v[e] > 0.0f ? v[e] : 0.0f;
        return v;
    }, acc);
    post_tiles<MT, NT>(red, acc, wave, lane);
    for (int i = wave; i < MT; i += RNNT_WK) {
        const int b = (blockIdx.y * MT + i) * 16 + r16;
        unsigned long long k = 0;
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const f32x4_t v = sum_waves<MT, NT>(red, j * MT + i, lane);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int c = (blockIdx.x * NT + j) * 16 + 4 * q + e;
                if (c >= V) continue;
                const float x = bias[c] + v[e];
                if (x > -INFINITY) k = max(k, (unsigned long long)ordered_bits(x) << 32 | (0xffffffffu - (uint32_t)c));
            }
        }
        k = max(k, __shfl_xor(k, 16));
        k = max(k, __shfl_xor(k, 32));
        // (the old value is waited for, so the maximum is posted before the barrier below; an agent-scope
        // fence would write back the L2 instead: 13.0 us a launch of the joint at one row, 6.6 this way)
        if (q == 0 && b < n && k != 0) {
            const unsigned long long old = atomicMax(key + b, k);
            asm volatile("" : : "v"(old) : "memory");
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) is_last = atomicAdd(done, 1u) == gridDim.x * gridDim.y - 1;
    __syncthreads();
    if (!is_last) return;
    for (int b = threadIdx.x; b < n; b += blockDim.x) {
        const unsigned long long k = atomicExch(key + b, 0ull);
        best[b] = k == 0 ? -1 : (int32_t)(0xffffffffu - (uint32_t)k);
    }
    if (threadIdx.x == 0) atomicExch(done, 0u);
}

}  // namespace ud

using namespace ud;

static int rfail(int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    return ud_set_error(code, buf);
}

#define RHIPC(call)                                                                              \
    do {                                                                                         \
        hipError_t e_ = (call);                                                                  \
        if (e_ != hipSuccess) return rfail(UD_ERR_HIP, "%s: %s", #call, hipGetErrorString(e_));  \
    } while (0)
#define RLAUNCH(what)                                                                            \
    do {                                                                                         \
        hipError_t e_ = hipGetLastError();                                                       \
        if (e_ != hipSuccess) return rfail(UD_ERR_HIP, "%s: launch failed: %s", what, hipGetErrorString(e_)); \
    } while (0)

enum RSlot { R_EMBED, R_PRED_W, R_PRED_B, R_OUT_W, R_OUT_B, R_ENC_W, R_ENC_B, R_FIXED };

struct ud_rnnt {
    int H, V, L, E, S, max_sym;
    float* w[R_FIXED] = {};                     // the product matrices fragment-major (frag_index_f32)
    int Vp;                                     // V rounded up to whole 64-column tiles (zero rows)
    std::vector<float*> wcat, bias;             // per layer [4H][2H] = [W_ih | W_hh] (unit-major rows,
                                                // rnnt_lstm_kernel), b_ih + b_hh
    std::vector<std::vector<float>> ih, hh, bih, bhh;   // host copies until both halves are set
    uint32_t set_fixed = 0;
    std::vector<uint32_t> set_layer;            // bit 0..3: weight_ih, weight_hh, bias_ih, bias_hh
    // h and c of each slot's two states [2][S][L][H] (state flip[slot] is the committed one, the other
    // the one its cached prediction leaves), the cached prediction's joint.pred output pg [S][H]
    float *h = nullptr, *c = nullptr, *pg = nullptr;
    std::vector<int> last, pending, flip;
    // the joint's row maxima (one key per (stream, frame) pair, grown to the largest call) and the
    // count of finished workgroups: zero between launches
    unsigned long long* key = nullptr;
    unsigned int* done = nullptr;
    int cap_pairs = 0;
    // A greedy iteration's lists, packed and uploaded in one copy from a pinned mirror: [slots to
    // predict][their last tokens][their state flips][joint rows' slots][joint rows' proj rows],
    // 3 S + 2 cap_pairs entries.  The host rewrites the mirror only after the iteration's
    // synchronize, when the previous copy from it is done.
    int32_t *dlist = nullptr, *hlist = nullptr;
    // the joint's argmax per row: pinned, mapped host memory the argmax kernel writes (dbest is its
    // device address), read after the iteration's synchronize
    int32_t *hbest = nullptr, *dbest = nullptr;
    // Work order across HIP streams (the calls share the workspaces above): every call that
    // enqueues device work records done_ev on its stream at its end, and a call on a different
    // stream first makes its stream wait for done_ev, so calls run in call order.
    hipEvent_t done_ev = nullptr;
    hipStream_t last_st = nullptr;
    bool has_last = false;
};

static float* ralloc(size_t floats) {
    void* p = nullptr;
    if (hipMalloc(&p, floats ? floats * 4 : 16) != hipSuccess) return nullptr;
    return static_cast<float*>(p);
}

static void free_rnnt(ud_rnnt* r) {
    if (!r) return;
    (void)hipDeviceSynchronize();
    for (float* p : r->w) if (p) (void)hipFree(p);
    for (float* p : r->wcat) if (p) (void)hipFree(p);
    for (float* p : r->bias) if (p) (void)hipFree(p);
    void* ps[] = {r->h, r->c, r->pg, r->key, r->done, r->dlist};
    for (void* p : ps) if (p) (void)hipFree(p);
    for (void* p : {(void*)r->hlist, (void*)r->hbest})
        if (p) (void)hipHostFree(p);
    if (r->done_ev) (void)hipEventDestroy(r->done_ev);
    delete r;
}

extern "C" UD_API int ud_rnnt_create(int32_t hidden, int32_t vocab, int32_t layers, int32_t enc_dim,
                                     int32_t max_streams, int32_t max_symbols_per_frame, ud_rnnt** out) {
    if (!out) return rfail(UD_ERR_INVALID, "ud_rnnt_create: null out pointer");
    *out = nullptr;
    if (hidden < 1 || vocab < 2 || layers < 1 || layers > 8 || enc_dim < 1 || max_streams < 1 || max_symbols_per_frame < 1)
        return rfail(UD_ERR_SHAPE, "ud_rnnt_create: bad dimensions");
    if (hidden % 64 != 0 || enc_dim % 16 != 0)
        return rfail(UD_ERR_SHAPE, "ud_rnnt_create: hidden %d must be a multiple of 64 and enc_dim %d of 16", hidden, enc_dim);
    ud_rnnt* r = new ud_rnnt();
    r->H = hidden; r->V = vocab; r->L = layers; r->E = enc_dim; r->S = max_streams; r->max_sym = max_symbols_per_frame;
    const size_t H = hidden, L = layers, S = max_streams;
    r->wcat.assign(L, nullptr);
    r->bias.assign(L, nullptr);
    r->ih.resize(L); r->hh.resize(L); r->bih.resize(L); r->bhh.resize(L);
    r->set_layer.assign(L, 0);
    r->Vp = (vocab + 63) / 64 * 64;
    bool ok = (r->h = ralloc(2 * S * L * H)) && (r->c = ralloc(2 * S * L * H)) && (r->pg = ralloc(S * H)) &&
              (r->done = (unsigned int*)ralloc(1)) && hipMemset(r->done, 0, sizeof(unsigned int)) == hipSuccess &&
              hipEventCreateWithFlags(&r->done_ev, hipEventDisableTiming) == hipSuccess;
    if (!ok || hipMemset(r->h, 0, 2 * S * L * H * 4) != hipSuccess || hipMemset(r->c, 0, 2 * S * L * H * 4) != hipSuccess) {
        free_rnnt(r);
        return rfail(UD_ERR_NOMEM, "ud_rnnt_create: device allocation failed");
    }
    r->last.assign(S, vocab - 1);
    r->pending.assign(S, 0);
    r->flip.assign(S, 0);
    *out = r;
    return UD_OK;
}

extern "C" UD_API void ud_rnnt_destroy(ud_rnnt* r) { free_rnnt(r); }

static int rupload(float*& dst, const float* src, size_t n) {
    if (!dst && !(dst = ralloc(n))) return rfail(UD_ERR_NOMEM, "ud_rnnt_set_weight: allocation failed");
    RHIPC(hipMemcpy(dst, src, n * 4, hipMemcpyHostToDevice));
    return UD_OK;
}

// A [rows, cols] matrix in the products' layout, with zero rows up to rows_padded.
static int rupload_frag(float*& dst, const float* src, int64_t rows, int64_t rows_padded, int64_t cols) {
    std::vector<float> t((size_t)rows_padded * cols, 0.0f);
    for (int64_t r = 0; r < rows; r++)
        for (int64_t c = 0; c < cols; c += 4) memcpy(&t[(size_t)frag_index_f32(r, (int)c, (int)(cols / 16))], src + r * cols + c, 16);
    return rupload(dst, t.data(), t.size());
}

extern "C" UD_API int ud_rnnt_get_info(const ud_rnnt* r, int32_t* hidden, int32_t* vocab, int32_t* layers,
                                       int32_t* enc_dim, int32_t* max_streams, int32_t* max_symbols_per_frame) {
    if (!r) return rfail(UD_ERR_INVALID, "ud_rnnt_get_info: null decoder");
    if (hidden) *hidden = r->H;
    if (vocab) *vocab = r->V;
    if (layers) *layers = r->L;
    if (enc_dim) *enc_dim = r->E;
    if (max_streams) *max_streams = r->S;
    if (max_symbols_per_frame) *max_symbols_per_frame = r->max_sym;
    return UD_OK;
}

extern "C" UD_API int ud_rnnt_set_weight(ud_rnnt* r, const char* name, const float* host, int64_t count) {
    if (!r || !name || !host) return rfail(UD_ERR_INVALID, "ud_rnnt_set_weight: null argument");
    const int64_t H = r->H, V = r->V, E = r->E;
    struct Fixed { const char* n; int slot; int64_t count; };
    const Fixed fixed[] = {{"decoder.prediction.embed.weight", R_EMBED, V * H}, {"joint.pred.weight", R_PRED_W, H * H},
                           {"joint.pred.bias", R_PRED_B, H}, {"joint.joint_net.2.weight", R_OUT_W, V * H},
                           {"joint.joint_net.2.bias", R_OUT_B, V}, {"joint.enc.weight", R_ENC_W, H * E},
                           {"joint.enc.bias", R_ENC_B, H}};
    for (const Fixed& f : fixed) {
        if (strcmp(name, f.n) != 0) continue;
        if (count != f.count)
            return rfail(UD_ERR_WEIGHT, "weight '%s': %lld values, expected %lld", name, (long long)count, (long long)f.count);
        const bool matrix = f.slot == R_PRED_W || f.slot == R_OUT_W || f.slot == R_ENC_W;
        int rc = !matrix ? rupload(r->w[f.slot], host, (size_t)count)
                         : rupload_frag(r->w[f.slot], host, f.slot == R_OUT_W ? V : H, f.slot == R_OUT_W ? r->Vp : H,
                                        f.slot == R_ENC_W ? E : H);
        if (rc == UD_OK) r->set_fixed |= 1u << f.slot;
        return rc;
    }
    const char* pre = "decoder.prediction.dec_rnn.lstm.";
    if (strncmp(name, pre, strlen(pre)) == 0) {
        const char* p = name + strlen(pre);
        const char* kinds[4] = {"weight_ih_l", "weight_hh_l", "bias_ih_l", "bias_hh_l"};
        for (int k = 0; k < 4; k++) {
            const size_t kl = strlen(kinds[k]);
            if (strncmp(p, kinds[k], kl) != 0) continue;
            char* end = nullptr;
            const long l = strtol(p + kl, &end, 10);
            if (end == p + kl || *end != '\0' || l < 0 || l >= r->L) break;
            const int64_t want = k < 2 ? 4 * H * H : 4 * H;
            if (count != want)
                return rfail(UD_ERR_WEIGHT, "weight '%s': %lld values, expected %lld", name, (long long)count, (long long)want);
            std::vector<float>& dst = k == 0 ? r->ih[l] : k == 1 ? r->hh[l] : k == 2 ? r->bih[l] : r->bhh[l];
            dst.assign(host, host + count);
            r->set_layer[l] |= 1u << k;
            int rc = UD_OK;
            if ((r->set_layer[l] & 3u) == 3u) {     // both matrices: [4H][2H] = [W_ih | W_hh], unit-major
                std::vector<float> cat((size_t)4 * H * 2 * H);
                for (int64_t g = 0; g < 4; g++)
                    for (int64_t j = 0; j < H; j++) {
                        float* row = &cat[(size_t)(4 * j + g) * 2 * H];
                        memcpy(row, &r->ih[l][(size_t)(g * H + j) * H], (size_t)H * 4);
                        memcpy(row + H, &r->hh[l][(size_t)(g * H + j) * H], (size_t)H * 4);
                    }
                rc = rupload_frag(r->wcat[l], cat.data(), 4 * H, 4 * H, 2 * H);
            }
            if (rc == UD_OK && (r->set_layer[l] & 12u) == 12u) {
                std::vector<float> b((size_t)4 * H);
                for (int64_t i = 0; i < 4 * H; i++) b[i] = r->bih[l][i] + r->bhh[l][i];
                rc = rupload(r->bias[l], b.data(), b.size());
            }
            return rc;
        }
    }
    return rfail(UD_ERR_WEIGHT, "unknown RNN-T weight name '%s'", name);
}

static int check_weights(const ud_rnnt* r, const char* who) {
    if (r->set_fixed != (1u << R_FIXED) - 1) return rfail(UD_ERR_STATE, "%s: joint / embedding weights not all set", who);
    for (int l = 0; l < r->L; l++)
        if (r->set_layer[l] != 15u) return rfail(UD_ERR_STATE, "%s: LSTM layer %d weights not all set", who, l);
    return UD_OK;
}

extern "C" UD_API int ud_rnnt_reset(ud_rnnt* r, int32_t slot) {
    if (!r) return rfail(UD_ERR_INVALID, "ud_rnnt_reset: null decoder");
    if (slot < 0 || slot >= r->S) return rfail(UD_ERR_SHAPE, "ud_rnnt_reset: slot %d outside 0..%d", slot, r->S - 1);
    const size_t LH = (size_t)r->L * r->H;
    RHIPC(hipMemset(r->h + slot * LH, 0, LH * 4));
    RHIPC(hipMemset(r->c + slot * LH, 0, LH * 4));
    r->last[slot] = r->V - 1;
    r->pending[slot] = 0;
    r->flip[slot] = 0;
    return UD_OK;
}

// The start of a call that enqueues device work on `st`: after every earlier call's work.
static int order_after_last(ud_rnnt* r, hipStream_t st) {
    if (r->has_last && st != r->last_st) RHIPC(hipStreamWaitEvent(st, r->done_ev, 0));
    return UD_OK;
}
// The end of such a call: done_ev marks the end of its work.
static int mark_done(ud_rnnt* r, hipStream_t st) {
    RHIPC(hipEventRecord(r->done_ev, st));
    r->last_st = st;
    r->has_last = true;
    return UD_OK;
}

static StateAt state_of(const ud_rnnt* r) { return StateAt{r->h, r->c, (int64_t)r->S * r->L * r->H, r->L, r->H}; }

// Row blocks of MT 16-row tiles, one, two or four by the rows there are (each workgroup's weights pass
// by MT row tiles); from 256 rows on also NT column tiles per workgroup, so that the rows are read less
// often.
template <int MT, int NT>
static void linear_tile(const float* W, const float* bias, const float* x, const int32_t* slot, const int32_t* flip,
                        StateAt sa, float* out, int n, int N, int K, hipStream_t st) {
    hipLaunchKernelGGL((rnnt_linear_kernel<MT, NT>), dim3(N / (16 * NT), (n + 16 * MT - 1) / (16 * MT)), dim3(64 * RNNT_WK), 0,
                       st, W, bias, x, slot, flip, sa, out, n, N, K);
}
static void launch_linear(const float* W, const float* bias, const float* x, const int32_t* slot, const int32_t* flip,
                          StateAt sa, float* out, int n, int N, int K, hipStream_t st) {
    if (n <= 16) linear_tile<1, 1>(W, bias, x, slot, flip, sa, out, n, N, K, st);
    else if (n <= 32) linear_tile<2, 1>(W, bias, x, slot, flip, sa, out, n, N, K, st);
    else if (n <= 256) linear_tile<4, 1>(W, bias, x, slot, flip, sa, out, n, N, K, st);
    else linear_tile<4, 4>(W, bias, x, slot, flip, sa, out, n, N, K, st);
}

extern "C" UD_API int ud_rnnt_project(ud_rnnt* r, int32_t rows, const float* enc_dev, float* out_dev, void* hip_stream) {
    if (!r || !enc_dev || !out_dev) return rfail(UD_ERR_INVALID, "ud_rnnt_project: null argument");
    if (!(r->set_fixed & (1u << R_ENC_W)) || !(r->set_fixed & (1u << R_ENC_B)))
        return rfail(UD_ERR_STATE, "ud_rnnt_project: joint.enc weights not set");
    if (rows < 1) return rfail(UD_ERR_SHAPE, "ud_rnnt_project: rows must be >= 1");
    if (reinterpret_cast<uintptr_t>(enc_dev) & 15 || (rows + 63) / 64 > 65535)
        return rfail(UD_ERR_SHAPE, "rnnt GEMM launch failed (%d x %d x %d)", rows, r->H, r->E);
    hipStream_t st = static_cast<hipStream_t>(hip_stream);
    int rc = order_after_last(r, st);
    if (rc != UD_OK) return rc;
    launch_linear(r->w[R_ENC_W], r->w[R_ENC_B], enc_dev, nullptr, nullptr, state_of(r), out_dev, rows, r->H, r->E, st);
    RLAUNCH("ud_rnnt_project");
    return mark_done(r, st);
}

template <int MT>
static void lstm_tile(const ud_rnnt* r, int n, const int32_t* dl, int layer, hipStream_t st) {
    hipLaunchKernelGGL(rnnt_lstm_kernel<MT>, dim3(r->H / 4, (n + 16 * MT - 1) / (16 * MT)), dim3(64 * RNNT_WK), 0, st,
                       r->wcat[layer], r->bias[layer], r->w[R_EMBED], dl, dl + n, dl + 2 * n, state_of(r), n, layer, r->V - 1);
}

// The prediction network for n slots without a cached prediction.  dl: the slots on the device, then
// their last tokens, then their state flips (uploaded with the iteration's lists).
static int predict(ud_rnnt* r, int n, const int32_t* dl, hipStream_t st) {
    for (int l = 0; l < r->L; l++) {
        if (n <= 16) lstm_tile<1>(r, n, dl, l, st);
        else if (n <= 32) lstm_tile<2>(r, n, dl, l, st);
        else lstm_tile<4>(r, n, dl, l, st);
        RLAUNCH("rnnt lstm");
    }
    launch_linear(r->w[R_PRED_W], r->w[R_PRED_B], r->h, dl, dl + 2 * n, state_of(r), r->pg, n, r->H, r->H, st);
    RLAUNCH("rnnt joint.pred");
    return UD_OK;
}

template <int MT, int NT>
static void joint_tile(const ud_rnnt* r, int n, const float* proj, const int32_t* dq, hipStream_t st) {
    hipLaunchKernelGGL((rnnt_joint_kernel<MT, NT>), dim3((r->V + 16 * NT - 1) / (16 * NT), (n + 16 * MT - 1) / (16 * MT)),
                       dim3(64 * RNNT_WK), 0, st, r->w[R_OUT_W], r->w[R_OUT_B], proj, r->pg, dq, dq + n, r->key, r->done,
                       r->dbest, n, r->V, r->H);
}

// Grows the joint's pair workspace to P rows.  Called between greedy calls only (every call ends
// with a stream synchronize), so nothing in flight uses the old buffers.
static int ensure_pairs(ud_rnnt* r, int P) {
    if (P <= r->cap_pairs) return UD_OK;
    void* ds[] = {r->key, r->dlist};
    for (void* p : ds) if (p) (void)hipFree(p);
    for (void* p : {(void*)r->hlist, (void*)r->hbest}) if (p) (void)hipHostFree(p);
    r->key = nullptr;
    r->dlist = r->hlist = r->hbest = r->dbest = nullptr;
    r->cap_pairs = 0;
    const size_t n = (size_t)P, nl = 3 * (size_t)r->S + 2 * n;
    bool ok = (r->key = (unsigned long long*)ralloc(2 * n)) && hipMemset(r->key, 0, n * 8) == hipSuccess &&
              (r->dlist = (int32_t*)ralloc(nl)) && hipHostMalloc((void**)&r->hlist, nl * 4) == hipSuccess &&
              hipHostMalloc((void**)&r->hbest, n * 4, hipHostMallocMapped | hipHostMallocCoherent) == hipSuccess &&
              hipHostGetDevicePointer((void**)&r->dbest, r->hbest, 0) == hipSuccess && hipStreamSynchronize(0) == hipSuccess;
    if (!ok) return rfail(UD_ERR_NOMEM, "ud_rnnt_greedy: joint workspace allocation failed (%d pairs)", P);
    r->cap_pairs = P;
    return UD_OK;
}

// Greedy decoding with speculative frames.  The sequential rule (RNNT.swift:125-151) evaluates the
// joint at (frame t, current prediction); a blank moves to t + 1 with the prediction unchanged.  So
// for each active stream one iteration evaluates the joint at EVERY remaining frame of the call
// (up to RNNT_SPEC of them) under the current prediction, and the host walks the results: leading
// blanks advance the frame, the first non-blank is emitted (its frame's symbol count continues
// from the previous emissions there), and later results of that stream are discarded because the
// prediction changes.  Every decision is the one the sequential loop makes; a chunk whose frames
// are all blank costs one iteration instead of one per frame.
constexpr int RNNT_SPEC = 16;

extern "C" UD_API int ud_rnnt_greedy(ud_rnnt* r, int32_t n, const int32_t* slots_host, const float* proj_dev,
                                     int32_t rows_per_stream, const int32_t* frames_host, int32_t* tokens_host,
                                     int32_t cap, int32_t* n_tokens_host, void* hip_stream) {
    if (!r || !slots_host || !proj_dev || !frames_host || !n_tokens_host || (cap > 0 && !tokens_host))
        return rfail(UD_ERR_INVALID, "ud_rnnt_greedy: null argument");
    int rc = check_weights(r, "ud_rnnt_greedy");
    if (rc != UD_OK) return rc;
    if (n < 1 || n > r->S) return rfail(UD_ERR_SHAPE, "ud_rnnt_greedy: n = %d outside 1..%d", n, r->S);
    std::vector<char> seen(r->S, 0);
    int max_frames = 0;
    for (int b = 0; b < n; b++) {
        const int s = slots_host[b];
        if (s < 0 || s >= r->S || seen[s]) return rfail(UD_ERR_INVALID, "ud_rnnt_greedy: bad or repeated slot %d", s);
        seen[s] = 1;
        if (frames_host[b] < 0 || frames_host[b] > rows_per_stream)
            return rfail(UD_ERR_SHAPE, "ud_rnnt_greedy: frames %d outside 0..%d", frames_host[b], rows_per_stream);
        if (frames_host[b] > max_frames) max_frames = frames_host[b];
        n_tokens_host[b] = 0;
    }
    hipStream_t st = static_cast<hipStream_t>(hip_stream);
    if ((rc = order_after_last(r, st)) != UD_OK) return rc;
    if ((rc = ensure_pairs(r, n * std::min(max_frames, RNNT_SPEC))) != UD_OK) return rc;
    const int V = r->V, blank = V - 1;
    std::vector<int> act, t(n, 0), em(n, 0), p0(n), p1(n);
    int32_t* hl = r->hlist;
    for (;;) {
        act.clear();
        for (int b = 0; b < n; b++)
            if (t[b] < frames_host[b]) act.push_back(b);
        if (act.empty()) break;
        int m = 0;
        for (int b : act) {
            p0[b] = m;
            m += std::min(frames_host[b], t[b] + RNNT_SPEC) - t[b];
            p1[b] = m;
        }
        if ((m + 63) / 64 > 65535) return rfail(UD_ERR_SHAPE, "ud_rnnt_greedy: %d joint rows beyond the grid", m);
        // one upload: predictions (slots, last tokens, state flips), joint rows (slots, proj rows)
        int np = 0;
        for (int b : act) np += r->pending[slots_host[b]] ? 0 : 1;
        int32_t *hp = hl, *hq = hl + 3 * np;
        for (int b : act) {
            const int s = slots_host[b];
            if (!r->pending[s]) {
                hp[0] = s;
                hp[np] = r->last[s];
                hp[2 * np] = r->flip[s];
                hp++;
            }
            for (int p = p0[b]; p < p1[b]; p++) {
                hq[p] = s;
                hq[m + p] = b * rows_per_stream + t[b] + (p - p0[b]);
            }
        }
        RHIPC(hipMemcpyAsync(r->dlist, hl, (size_t)(3 * np + 2 * m) * 4, hipMemcpyHostToDevice, st));
        if (np && (rc = predict(r, np, r->dlist, st)) != UD_OK) return rc;
        for (int b : act) r->pending[slots_host[b]] = 1;
        const int32_t* dq = r->dlist + 3 * np;
        if (m <= 16) joint_tile<1, 1>(r, m, proj_dev, dq, st);
        else if (m <= 32) joint_tile<2, 1>(r, m, proj_dev, dq, st);
        else if (m <= 256) joint_tile<4, 1>(r, m, proj_dev, dq, st);
        else joint_tile<4, 4>(r, m, proj_dev, dq, st);
        RLAUNCH("rnnt joint");
        RHIPC(hipStreamSynchronize(st));
        for (int b : act) {
            const int s = slots_host[b];
            for (int p = p0[b]; p < p1[b]; p++) {
                const int tt = t[b], k = r->hbest[p];
                if (k == blank || k < 0 || k >= V) {   // (out of range only for NaN logits)
                    t[b] = tt + 1;
                    em[b] = 0;
                    continue;
                }
                if (n_tokens_host[b] < cap) tokens_host[(int64_t)b * cap + n_tokens_host[b]] = k;
                n_tokens_host[b]++;
                r->last[s] = k;             // the cached prediction's state becomes the committed one
                r->pending[s] = 0;
                r->flip[s] ^= 1;
                if (++em[b] >= r->max_sym) {
                    t[b] = tt + 1;
                    em[b] = 0;
                }
                break;
            }
        }
    }
    if (max_frames == 0) RHIPC(hipStreamSynchronize(st));   // (else the last iteration did)
    return mark_done(r, st);
}
