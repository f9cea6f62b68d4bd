// GEMMs of the encoder step, C = epilogue(A[M,K] . W[N,K]^T), W in the checkpoint's [out, in]
// orientation (Sources/DictatorEngine/Core/Kernels.swift:79-112; epilogue order of
// Sources/DictatorEngine/Metal/12_gemm2.metal:111-122: act, then out_scale, then + residual).
//
// 16-bit path: v_mfma_f32_16x16x32_f16 (gfx950) on IEEE-half operands.  The streaming step multiplies
// M = streams x T rows (128 at 64 streams x 2 frames) against 2-8 MB weight matrices.  Measured on
// MI355X, the limit at few rows is not HBM but the L2 -> CU traffic of the activation fragments, which
// every column tile re-reads; so both operands are stored fragment-major (see frag_index): each
// operand fragment is one contiguous 1 KB load, with no partially used cache lines.
//  - gemm_bf16_kernel, few rows: each wave owns a [16*MT x 16*NT] output tile (shapes per GEMM in
//    launch_few) and every WK-th 64-wide K chunk of its workgroup's K range; the WK waves are summed
//    in LDS; two register buffers, separated by scheduling barriers, keep the next chunk's loads in
//    flight behind the current chunk's MFMAs;
//  - gemm_panel_kernel, many rows: the waves of a workgroup share a row panel through LDS and each
//    stream their own weights;
//  - plan16 chooses between them;
//  - ksplit > 1 splits K over workgroups (parallelism for the N = 1024 projections); each split
//    writes its own fp32 partial slab and the following LayerNorm adds the slabs, in order, to the
//    residual row it reads anyway -- deterministic, no atomics, no extra kernel.
// Epilogues: act + half store (row-major, or fragment-major for a following GEMM), fp32 store,
// split-K partial slabs, and the QKV projection's split store:
// q row-major into the buffer the attention reads, K and V straight into their K/V ring rows (so
// the new rows are written once, and the attention kernel only reads the rings).
#include <type_traits>

#include "ud_common.hpp"
#include "kernels.hpp"

namespace ud {

// Maps the linear workgroup id so that tiles t, t+1, ... of one XCD's share are contiguous
// (workgroups are dealt round-robin to the 8 XCDs): the M tiles and K splits of one N tile then
// run on the same XCD and share its L2.
__device__ __forceinline__ int xcd_tile(int bid, int total) {
    if (total % 8 != 0) return bid;
    return (bid % 8) * (total / 8) + bid / 8;
}

// The 16-bit K/V ring element of a QKV projection output in column n of [D, 3D), for an output row
// whose ring row starts at element rowoff of the slot's head-0 block (QkvRing::rows): K for
// n < 2D, V above, head (n - D) mod D / 128.
__device__ __forceinline__ uint16_t* qkv_ring_dst(const QkvRing& r, int rowoff, int n) {
    const int D = r.H * 128;
    const int c = n - D, part = c >= D ? 1 : 0, cc = c - part * D;
    uint16_t* base = static_cast<uint16_t*>(part ? r.vring : r.kring);
    return base + rowoff + (int64_t)(cc >> 7) * r.R * 128 + (cc & 127);
}

// 16 bytes of the QKV ring-row table per lane, global -> LDS at dst + 16 * lane (a plain function:
// the builtin written in a kernel template's body drops the host stub of some instantiations).
__device__ __forceinline__ void lds_direct16_rows(const int32_t* src, int32_t* dst) {
    __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0);
}

// EPI_SUBFLAT: the out Linear's A-operand element of GEMM row m, column n (-1: row not stored), and
// whether the row is masked (written as zero).
__device__ __forceinline__ int64_t subflat_dst(const GemmArgs& a, int64_t m, int n, bool& masked) {
    const SubFlat& f = a.flat;
    const int per = f.T3 * f.F3, mi = (int)m;                 // M < 2^31 (launch_gemm)
    const int s = mi / per, rem = mi - s * per, t3 = rem / f.F3, f3 = rem - t3 * f.F3;
    masked = t3 >= f.vlen[4 * s + 3];
    if (t3 < f.drop) return -1;
    return frag_index((int64_t)s * f.T + t3 - f.drop, f3 * a.N + n, f.F3 * a.N / 64);
}

// Four floats as IEEE half, packed.
__device__ __forceinline__ uint2 pack4(float x, float y, float z, float w) {
    return make_uint2((uint32_t)f2h(x) | ((uint32_t)f2h(y) << 16), (uint32_t)f2h(z) | ((uint32_t)f2h(w) << 16));
}

template <int MT, int NT>
struct Frag {
    uint4 a[MT][2];
    uint4 b[NT][2];
};

template <int MT, int NT>
__device__ __forceinline__ void load_frag(Frag<MT, NT>& f, const bf16* const* ap, const bf16* const* wp, int64_t off) {
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        f.a[mt][0] = ld16(ap[mt] + off);
        f.a[mt][1] = ld16(ap[mt] + off + 512);
    }
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        f.b[nt][0] = ld16(wp[nt] + off);
        f.b[nt][1] = ld16(wp[nt] + off + 512);
    }
}

template <int MT, int NT>
__device__ __forceinline__ void mma_frag(const Frag<MT, NT>& f, f32x4_t (&acc)[NT][MT]) {
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
                acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_f16x8(f.a[mt][h]), as_f16x8(f.b[nt][h]),
                                                                     acc[nt][mt], 0, 0, 0);
}

// Grid: (N/16) x ceil(M/(16*MT)) x ksplit workgroups of WK waves.  The host guarantees
// K % (64 * ksplit) == 0 and at least WK 64-deep chunks per split: wave w takes chunks w, w + WK,
// .. of its split, so when WK does not divide the chunk count the first waves take one more.  The epilogue kind and activation are template parameters: a
// runtime-switched, fully unrolled epilogue measured ~3.5 us slower per launch on MI355X (its
// code does not stay in the instruction cache).
template <int MT, int WK, int EPI, int ACT, int NT, bool BIAS = false>
__global__ __launch_bounds__(64 * WK, 1) void gemm_bf16_kernel(GemmArgs a) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int nN = a.N / (16 * NT), nM = (a.M + 16 * MT - 1) / (16 * MT);
    const int ks = a.ksplit;
    const int t = xcd_tile(blockIdx.x, nN * nM * ks);
    const int kz = t % ks, tile = t / ks;
    const int nt = tile / nM, mb = tile % nM;
    const int nk = a.K / 64;
    const int kper = nk / ks;
    const int kc0 = kz * kper + wave;
    const int rtiles = (a.M + 15) / 16;

    const bf16* A = static_cast<const bf16*>(a.A);
    const bf16* W = static_cast<const bf16*>(a.W);
    // QKV split store: the ring offsets of the workgroup's 16 MT rows, into LDS (read in the
    // epilogue, after the workgroup barrier); the table is padded past the last row
    __shared__ __attribute__((aligned(16))) int32_t rtab[EPI == EPI_QKV_RING ? 16 * MT : 4];
    if constexpr (EPI == EPI_QKV_RING) {
        if (wave == 0 && lane < 4 * MT)
            lds_direct16_rows(a.ring.rows + mb * 16 * MT + 4 * lane, rtab);
    }
    const bf16* ap[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const int rt = min(mb * MT + mt, rtiles - 1);      // clamped tiles are computed, not stored
        ap[mt] = A + (((int64_t)rt * nk + kc0) << 10) + lane * 8;
    }
    const bf16* wp[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) wp[j] = W + (((int64_t)(nt * NT + j) * nk + kc0) << 10) + lane * 8;

    f32x4_t acc[NT][MT];
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[j][mt] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    const int cnt = (kper - wave + WK - 1) / WK;   // chunks of this wave (>= 1)
    constexpr int STEP = WK * 1024;       // element stride between a wave's consecutive chunks
    auto off = [&](int i) { return (int64_t)i * STEP; };
    Frag<MT, NT> f0, f1;
    load_frag(f0, ap, wp, off(0));
    int i = 0;
    for (; i + 2 < cnt; i += 2) {
        load_frag(f1, ap, wp, off(i + 1));
        __builtin_amdgcn_sched_barrier(0);
        mma_frag<MT, NT>(f0, acc);
        __builtin_amdgcn_sched_barrier(0);
        load_frag(f0, ap, wp, off(i + 2));
        __builtin_amdgcn_sched_barrier(0);
        mma_frag<MT, NT>(f1, acc);
        __builtin_amdgcn_sched_barrier(0);
    }
    if (i + 1 < cnt) {
        load_frag(f1, ap, wp, off(i + 1));
        __builtin_amdgcn_sched_barrier(0);
        mma_frag<MT, NT>(f0, acc);
        __builtin_amdgcn_sched_barrier(0);
        mma_frag<MT, NT>(f1, acc);
    } else {
        mma_frag<MT, NT>(f0, acc);
    }

    // Epilogue of one finished 16 x 16 accumulator (j, mt): the lane holds rows
    // 16*(mb*MT + mt) + 4*g + i (i < 4) of column 16*(nt*NT + j) + r16.
    auto finish = [&](int j, int mt, const f32x4_t& v4) {
        const int n = (nt * NT + j) * 16 + r16;
#pragma unroll
        for (int i2 = 0; i2 < 4; i2++) {
            const int64_t m = (int64_t)(mb * MT + mt) * 16 + g * 4 + i2;
            if (m >= a.M) continue;
            float v = v4[i2];
            if constexpr (BIAS) v += kz == 0 ? a.bias[n] : 0.0f;
            if constexpr (EPI == EPI_PARTIAL) {
                static_cast<float*>(a.C)[((int64_t)kz * a.M + m) * a.ldc + n] = a.out_scale * v;
            } else if constexpr (EPI == EPI_STORE_F32) {
                static_cast<float*>(a.C)[m * a.ldc + n] = apply_act(v, ACT) * a.out_scale;
            } else if constexpr (EPI == EPI_STORE_FRAG) {
                static_cast<uint16_t*>(a.C)[frag_index(m, n, a.N / 64)] = f2h(apply_act(v, ACT) * a.out_scale);
            } else if constexpr (EPI == EPI_QKV_RING) {
                const uint16_t x = f2h(apply_act(v, ACT) * a.out_scale);
                if (n < a.ring.H * 128) static_cast<uint16_t*>(a.C)[m * a.ldc + n] = x;
                else *qkv_ring_dst(a.ring, rtab[mt * 16 + g * 4 + i2], n) = x;
            } else if constexpr (EPI == EPI_SUBFLAT) {
                bool masked;
                const int64_t d = subflat_dst(a, m, n, masked);
                if (d >= 0) static_cast<uint16_t*>(a.C)[d] = masked ? (uint16_t)0 : f2h(apply_act(v, ACT) * a.out_scale);
            } else {
                static_cast<uint16_t*>(a.C)[m * a.ldc + n] = f2h(apply_act(v, ACT) * a.out_scale);
            }
        }
    };
    // EPI_GLU: accumulators j (values) and j + 1 (gates) of the same 16 channels; the lane's
    // channel is (nt NT / 2 + j / 2) * 16 + r16
    auto finish_glu = [&](int j, int mt, const f32x4_t& vv, const f32x4_t& vg) {
        const int c = (nt * NT / 2 + j / 2) * 16 + r16;
#pragma unroll
        for (int i2 = 0; i2 < 4; i2++) {
            const int64_t m = (int64_t)(mb * MT + mt) * 16 + g * 4 + i2;
            if (m >= a.M) continue;
            static_cast<uint16_t*>(a.C)[m * a.ldc + c] = f2h(vv[i2] * sigmoidf(vg[i2]));
        }
    };
    if constexpr (EPI == EPI_GLU) {
        static_assert(NT % 2 == 0, "value and gate tiles in pairs");
        if constexpr (WK > 1) {
            __shared__ f32x4_t red[WK][NT][MT][64];
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++) red[wave][j][mt][lane] = acc[j][mt];
            __syncthreads();
            for (int idx = wave; idx < NT / 2 * MT; idx += WK) {
                const int j = 2 * (idx / MT), mt = idx % MT;
                f32x4_t vv = red[0][j][mt][lane], vg = red[0][j + 1][mt][lane];
#pragma unroll
                for (int w = 1; w < WK; w++) { vv += red[w][j][mt][lane]; vg += red[w][j + 1][mt][lane]; }
                finish_glu(j, mt, vv, vg);
            }
        } else {
#pragma unroll
            for (int j = 0; j < NT; j += 2)
#pragma unroll
                for (int mt = 0; mt < MT; mt++) finish_glu(j, mt, acc[j][mt], acc[j + 1][mt]);
        }
        return;
    }
    if constexpr (WK > 1) {
        // Every wave parks its partial accumulators in LDS; wave w then finishes the accumulators
        // idx = j*MT + mt with idx % WK == w: the sum of the WK partials in wave order, and the
        // epilogue.  Spreading the sums and the stores over the waves keeps the workgroup's tail
        // short (one wave finishing every accumulator measured ~3 us per launch at 128 rows).
        __shared__ f32x4_t red[WK][NT][MT][64];
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++) red[wave][j][mt][lane] = acc[j][mt];
        if constexpr (EPI == EPI_QKV_RING) __builtin_amdgcn_s_waitcnt(0x0F70);   // the row table landed
        __syncthreads();
        for (int idx = wave; idx < NT * MT; idx += WK) {
            const int j = idx / MT, mt = idx % MT;
            f32x4_t v = red[0][j][mt][lane];
#pragma unroll
            for (int w = 1; w < WK; w++) v += red[w][j][mt][lane];
            finish(j, mt, v);
        }
    } else {
        if constexpr (EPI == EPI_QKV_RING) {
            __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): the row table's direct load landed
            __syncthreads();
        }
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++) finish(j, mt, acc[j][mt]);
    }
}

// ---------------------------------------------------------------- 16-bit, row panels through LDS
// A workgroup of NW waves owns a 16*MT x 16*NT*NW output tile.  Its waves stand side by side in N:
// wave w multiplies all 16*MT rows with its own 16*NT columns.  Per 32-deep K step
//  - the MT row fragments (1 KB half-blocks of the fragment-major layout, contiguous) go into an LDS
//    ring of four steps by direct global -> LDS loads and are read by every wave;
//  - each wave loads its own NT weight fragments straight into registers, three steps ahead: no two
//    waves of the workgroup read the same weights, so LDS would only add a pass.
// That split is what bounds the kernel: with both operands staged in LDS (256 x 256 or 224 x 256
// tiles, 8 waves of 112 or 128 x 64) a step read and wrote 88-128 KB of LDS per workgroup for 28-32
// MFMAs per wave, as long as the MFMAs themselves take; here a 112 x 256 tile moves 7 KB in and 28 KB
// out.  At 3,584 x 4,096 x 1,024 (random data, weights from HBM): 35.4 us with both operands in LDS,
// 30.9 us here (973 TFLOP/s); 1,024 x 4,096 x 1,024: 27.7 us (the register kernel that served these
// rows) -> 13.3.
//
// One barrier per step: at step s a wave waits until its own direct loads of step s have landed (those
// of s + 1 and s + 2 and the weights between them may be in flight), the barrier makes every wave's
// loads of s visible and says that every wave holds its step s - 1 fragments in registers, so the
// buffer of s - 1 takes the loads of s + 3.  Two workgroups per CU (or 8 waves) cover each other's
// barrier and LDS latency.  The four buffers are separate arrays and the loop is unrolled by four, so
// the compiler can tell them apart and does not wait for outstanding direct loads before LDS reads
// of another buffer.
//
// The MFMAs are inline asm with the accumulators pinned in place in the accumulator registers:
// compiled from the builtin, the register allocator moved accumulators between register files in the
// loop (and spilled them at 112 rows).  The compiler's hazard checks do not see inside the asm, so the
// required wait states are explicit at the two points where compiled code touches the accumulators;
// empty asm statements pin the zeroing before, and the epilogue's reads after, those waits.

// Buffer resource of `bytes` bytes at p: loads past them return zeros.  (Buffer loads rather than
// global ones: the compiler counts a global -> LDS load as one that may be flat, after which it waits
// for every outstanding load, not for the one it needs; and the step's offset is a scalar operand.)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_at(const void* p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}
// 16 bytes per lane from byte voff + soff of the buffer straight into LDS at dst + 16 * lane (dst
// wave-uniform).  (Plain functions: inside a lambda of a kernel template the host pass drops the
// kernel's stub.)
__device__ __forceinline__ void lds_buffer16(__amdgpu_buffer_rsrc_t r, int voff, int soff, bf16* dst) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, dst, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ uint4 ld_buffer16(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

template <int NT, int MT>
__device__ __forceinline__ void pin_acc(f32x4_t (&acc)[NT][MT]) {
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++) asm volatile("" : "+a"(acc[j][i]));
}

// The activation as a compile-time choice (silu is v_exp_f32 + v_rcp_f32, about 1 ulp each).
template <int ACT>
__device__ __forceinline__ float act_fast(float x) {
    if constexpr (ACT == ACT_SILU) return silu(x);
    else return apply_act(x, ACT);
}

// Row panels that consecutive workgroups of an XCD share before they move to the next columns: an
// XCD's 32 tiles then cover 4 row panels x 8 column panels, whose operands are a third of those of
// 1 x 32 (17.7 -> 16.7 us at 1,024 x 4,096 x 1,024, measured with both operands in LDS).
constexpr int PANEL_GROUP = 4;

template <int MT, int NT, int NW, int EPI, int ACT, bool BIAS>
__global__ __launch_bounds__(64 * NW, NW == 4 ? 2 : 1) void gemm_panel_kernel(GemmArgs a) {
    constexpr int TR = 16 * MT, BB = NT * NW;                // tile rows; W blocks (16 columns each) per tile
    constexpr int STAGE = MT * 512;                          // halves per LDS stage
    constexpr int CPS = (MT + NW - 1) / NW;                  // direct loads per wave per step
    __shared__ __attribute__((aligned(16))) bf16 st0[STAGE];
    __shared__ __attribute__((aligned(16))) bf16 st1[STAGE];
    __shared__ __attribute__((aligned(16))) bf16 st2[STAGE];
    __shared__ __attribute__((aligned(16))) bf16 st3[STAGE];
    __shared__ __attribute__((aligned(16))) int32_t rtab[EPI == EPI_QKV_RING ? TR : 4];    // QKV: ring row offsets
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int nN = a.N / (16 * BB), nM = (a.M + TR - 1) / TR;
    const int ks = a.ksplit;
    const int t = xcd_tile(blockIdx.x, nN * nM * ks);
    const int kz = t % ks, tile = t / ks;
    const int grp = tile / (PANEL_GROUP * nN), rem = tile - grp * PANEL_GROUP * nN;
    const int gm = min(PANEL_GROUP, nM - grp * PANEL_GROUP);
    const int mb = grp * PANEL_GROUP + rem % gm, nb = rem / gm;
    const int nk = a.K / 64, kper = nk / ks, kc0 = kz * kper;
    const int n = 2 * kper;                                  // 32-deep K steps of this split: a multiple of 4
    const int rtiles = (a.M + 15) / 16;
    const bf16* A = static_cast<const bf16*>(a.A);
    const bf16* W = static_cast<const bf16*>(a.W);
    const int lo = lane * 8;
    const int ct0 = (nb * NW + wave) * NT;                   // first column tile of this wave

    if constexpr (EPI == EPI_QKV_RING) {
        // the ring offsets of the tile's TR rows (the table is padded past the last row)
        for (int i = tid; i < TR; i += 64 * NW) rtab[i] = a.ring.rows[mb * TR + i];
    }
    // Wave w copies the row fragments w + NW j of each step (past the panel: its last one again) and
    // loads the column tiles ct0 + j.  Row tiles past the last one are clamped: computed, not stored.
    const int rt0 = mb * MT, rts = min(MT, rtiles - rt0);
    const __amdgpu_buffer_rsrc_t ra = buffer_at(A + (((int64_t)rt0 * nk + kc0) << 10), (rts * nk - kc0) * 2048);
    const __amdgpu_buffer_rsrc_t rw = buffer_at(W + (((int64_t)nb * BB * nk + kc0) << 10), (BB * nk - kc0) * 2048);
    int aoff[CPS], adst[CPS], woff[NT];
#pragma unroll
    for (int j = 0; j < CPS; j++) {
        const int u = min(wave + NW * j, MT - 1);
        aoff[j] = min(u, rts - 1) * nk * 2048;
        adst[j] = u * 512;
    }
#pragma unroll
    for (int j = 0; j < NT; j++) woff[j] = (wave * NT + j) * nk * 2048;

    uint4 w[4][NT], fa[MT];
    auto load_step = [&](int s, bf16* dst, uint4 (&wd)[NT]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < CPS; j++) lds_buffer16(ra, lane * 16, aoff[j] + s * 1024, dst + adst[j]);
#pragma unroll
        for (int j = 0; j < NT; j++) wd[j] = ld_buffer16(rw, lane * 16, woff[j] + s * 1024);
        __builtin_amdgcn_sched_barrier(0);
    };
    f32x4_t acc[NT][MT];
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++) acc[j][i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    // Step s in buffer cur; the loads of step s + 3 go to nxt / wn (LAST: there are none, and every
    // outstanding load is waited for).
    auto step = [&](int s, const bf16* cur, const uint4 (&wc)[NT], bf16* nxt, uint4 (&wn)[NT], auto last)
        __attribute__((always_inline)) {
        constexpr bool LAST = decltype(last)::value;
        // issued after this wave's direct loads of s: the weights of s, then the groups of s + 1, s + 2
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(LAST ? 0 : NT + 2 * (CPS + NT)));
        __builtin_amdgcn_s_barrier();
        __asm__ volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < MT; i++) fa[i] = *reinterpret_cast<const uint4*>(cur + i * 512 + lo);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!LAST) load_step(s + 3, nxt, wn);
        // (operands swapped, weights as the row operand: each 16 x 16 accumulator holds C^T, so a lane
        // has 4 consecutive output columns of one row)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int i = 0; i < MT; i++)
                asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0"
                             : "+a"(acc[j][i]) : "v"(as_f16x8(wc[j])), "v"(as_f16x8(fa[i])));
        __builtin_amdgcn_sched_barrier(0);
    };
    load_step(0, st0, w[0]);
    load_step(1, st1, w[1]);
    load_step(2, st2, w[2]);
    pin_acc(acc);
    asm volatile("s_nop 7");                                 // accumulator zeroing -> first MFMA
    const std::false_type more{};
    const std::true_type last{};
    int s = 0;
    for (; s + 4 < n; s += 4) {
        step(s, st0, w[0], st3, w[3], more);
        step(s + 1, st1, w[1], st0, w[0], more);
        step(s + 2, st2, w[2], st1, w[1], more);
        step(s + 3, st3, w[3], st2, w[2], more);
    }
    step(s, st0, w[0], st3, w[3], more);
    step(s + 1, st1, w[1], st0, w[0], last);
    step(s + 2, st2, w[2], st1, w[1], last);
    step(s + 3, st3, w[3], st2, w[2], last);
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7\n\ts_nop 7");   // last MFMA results -> epilogue reads
    pin_acc(acc);

    // acc[j][i] is tile (column tile j, row tile i) transposed: lane holds row 16*rt + r16 and the
    // 4 columns 16*ct + 4*g + e (e < 4).
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int64_t m = (int64_t)(mb * MT + i) * 16 + r16;
        if (m >= a.M) continue;
        if constexpr (EPI == EPI_GLU) {
            // column tiles j (values) and j + 1 (gates) of channels 8 (ct0 + j) ..
            static_assert(NT % 2 == 0, "value and gate tiles in pairs");
#pragma unroll
            for (int j = 0; j < NT; j += 2) {
                const int c = (ct0 + j) / 2 * 16 + g * 4;
                const f32x4_t vv = acc[j][i], vg = acc[j + 1][i];
                *reinterpret_cast<uint2*>(static_cast<bf16*>(a.C) + m * a.ldc + c) =
                    pack4(vv[0] * sigmoidf(vg[0]), vv[1] * sigmoidf(vg[1]), vv[2] * sigmoidf(vg[2]), vv[3] * sigmoidf(vg[3]));
            }
            continue;
        }
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const int c = (ct0 + j) * 16 + g * 4;
            f32x4_t v = acc[j][i];
            if constexpr (BIAS) v += *reinterpret_cast<const f32x4_t*>(a.bias + c);
            if constexpr (EPI == EPI_PARTIAL) {
                *reinterpret_cast<f32x4_t*>(static_cast<float*>(a.C) + ((int64_t)kz * a.M + m) * a.ldc + c) = v * a.out_scale;
                continue;
            }
            f32x4_t o;
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = act_fast<ACT>(v[e]) * a.out_scale;
            if constexpr (EPI == EPI_STORE_F32) {
                *reinterpret_cast<f32x4_t*>(static_cast<float*>(a.C) + m * a.ldc + c) = o;
            } else {
                uint2 h = pack4(o[0], o[1], o[2], o[3]);
                bf16* dst;
                if constexpr (EPI == EPI_QKV_RING) {   // 4 columns of one head: contiguous in the ring row
                    dst = c < a.ring.H * 128 ? static_cast<bf16*>(a.C) + m * a.ldc + c
                                             : qkv_ring_dst(a.ring, rtab[i * 16 + r16], c);
                } else if constexpr (EPI == EPI_SUBFLAT) {   // 4 columns: contiguous in the fragment block
                    bool masked;
                    const int64_t d = subflat_dst(a, m, c, masked);
                    if (d < 0) continue;
                    if (masked) h = make_uint2(0, 0);
                    dst = static_cast<bf16*>(a.C) + d;
                } else {
                    dst = static_cast<bf16*>(a.C) + (EPI == EPI_STORE_FRAG ? frag_index(m, c, a.N / 64) : m * a.ldc + c);
                }
                *reinterpret_cast<uint2*>(dst) = h;
            }
        }
    }
}

// ---------------------------------------------------------------- fp32 encoder (MFMA)
// The fp32 encoder's projections and front-end on v_mfma_f32_16x16x4_f32, shaped as gemm_bf16_kernel:
// a workgroup of 8 waves owns a 16*MT x 16*NT output tile and its waves take the 64-wide K chunks of
// the workgroup's K split in turn; the 8 partial tiles are summed in LDS in wave order.  At few rows
// the weights (92 MB a layer) bound it: they are stored fragment-major (frag_index_f32), so a wave
// streams 4 KB of contiguous weights per chunk, and with one 16-column tile per workgroup and 2-4 K
// splits of the N = 1024 projections 128-256 workgroups x 8 waves keep them in flight.  More rows
// take wider tiles (launch_f32), which re-read the activations less often.
// 8 rows: ff linear1 (4,096 x 1,024) 137 -> 5.9 us (2.8 TB/s), ff linear2 (1,024 x 4,096) 333 -> 5.9,
// linear_out (1,024 x 1,024) 333 (its launches averaged with linear2's) -> 4.5; the 64 x 64 VALU
// tiles before gave each CU at most one workgroup (16 for N = 1,024) that waited on every 16-wide K
// slice in turn.  24-layer step: 4 streams x 2 frames 45.9 -> 1.75 ms.
// Every output sums its K range in the same order whatever M is: a row's result does not depend on
// the batch it is computed in.
constexpr int F32_WK = 8;

// Fragments of half a K chunk (32 columns): two 16 x 16 blocks per tile.
template <int MT, int NT>
struct Frag32 {
    f32x4_t a[MT][2], b[NT][2];
};

template <int MT, int NT>
__device__ __forceinline__ void mma_frag32(const Frag32<MT, NT>& f, f32x4_t (&acc)[NT][MT]) {
#pragma unroll
    for (int g = 0; g < 2; g++)
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int i = 0; i < MT; i++)
                    acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.b[j][g][e], f.a[i][g][e], acc[j][i], 0, 0, 0);
}

template <int MT, int NT>
__global__ __launch_bounds__(64 * F32_WK) void gemm_f32_kernel(GemmArgs a) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, q = lane >> 4;
    const int nN = a.N / (16 * NT), nM = (a.M + 16 * MT - 1) / (16 * MT), ks = a.ksplit;
    const int t = xcd_tile(blockIdx.x, nN * nM * ks);
    const int kz = t % ks, tile = t / ks, nb = tile / nM, mb = tile % nM;
    const int nk = a.K / 64, kper = nk / ks, kc0 = kz * kper;
    const float* A = static_cast<const float*>(a.A);
    const float* W = static_cast<const float*>(a.W);
    // lane (r16, q): columns 4q .. 4q + 3 of row r16 of each 16 x 16 block; MFMA e takes element e of
    // both operands, so they see the same permutation of a block's 16 k values.  Rows past M repeat
    // the last one: computed, not stored.
    const float* ap[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) ap[i] = A + (int64_t)min((mb * MT + i) * 16 + r16, a.M - 1) * a.lda + kc0 * 64 + 4 * q;
    const float* wp[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) wp[j] = W + ((int64_t)(nb * NT + j) * nk + kc0) * 1024 + lane * 4;
    auto load = [&](Frag32<MT, NT>& f, int c, int h) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < 2; g++) {
#pragma unroll
            for (int j = 0; j < NT; j++) f.b[j][g] = *reinterpret_cast<const f32x4_t*>(wp[j] + (int64_t)c * 1024 + (2 * h + g) * 256);
#pragma unroll
            for (int i = 0; i < MT; i++) f.a[i][g] = *reinterpret_cast<const f32x4_t*>(ap[i] + c * 64 + (2 * h + g) * 16);
        }
    };
    f32x4_t acc[NT][MT];
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++) acc[j][i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    // chunks wave, wave + 8, ..; the next half chunk's loads are in flight behind this one's MFMAs
    Frag32<MT, NT> f0, f1;
    if (wave < kper) load(f0, wave, 0);
    for (int c = wave; c < kper; c += F32_WK) {
        load(f1, c, 1);
        __builtin_amdgcn_sched_barrier(0);
        mma_frag32<MT, NT>(f0, acc);
        __builtin_amdgcn_sched_barrier(0);
        if (c + F32_WK < kper) load(f0, c + F32_WK, 0);
        __builtin_amdgcn_sched_barrier(0);
        mma_frag32<MT, NT>(f1, acc);
        __builtin_amdgcn_sched_barrier(0);
    }
    // acc[j][i] holds C^T: the lane's row is r16 of row tile i, its columns 4q .. 4q + 3 of tile j
    __shared__ f32x4_t red[F32_WK][NT * MT][64];
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
        for (int i = 0; i < MT; i++) red[wave][j * MT + i][lane] = acc[j][i];
    __syncthreads();
    for (int idx = wave; idx < NT * MT; idx += F32_WK) {
        const int j = idx / MT, i = idx % MT;
        const int64_t m = (int64_t)(mb * MT + i) * 16 + r16;
        const int n = (nb * NT + j) * 16 + 4 * q;
        if (m >= a.M) continue;
        f32x4_t v = red[0][idx][lane];
#pragma unroll
        for (int w = 1; w < F32_WK; w++) v += red[w][idx][lane];
        if (a.bias != nullptr) v += *reinterpret_cast<const f32x4_t*>(a.bias + n);
        if (a.epi != EPI_PARTIAL) {
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = apply_act(v[e], a.act);
        }
        *reinterpret_cast<f32x4_t*>(static_cast<float*>(a.C) + ((int64_t)kz * a.M + m) * a.ldc + n) = v * a.out_scale;
    }
}

template <int MT, int NT>
static int launch_f32_tile(const GemmArgs& a, hipStream_t st) {
    const int tiles = a.N / (16 * NT) * ((a.M + 16 * MT - 1) / (16 * MT)) * a.ksplit;
    hipLaunchKernelGGL((gemm_f32_kernel<MT, NT>), dim3(tiles), dim3(64 * F32_WK), 0, st, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Row-major A, C and fragment-major W; EPI_STORE / EPI_STORE_F32 (with bias and activation) or
// EPI_PARTIAL slabs.
static int launch_f32(const GemmArgs& a, hipStream_t st) {
    const bool partial = a.epi == EPI_PARTIAL;
    if (!partial && a.epi != EPI_STORE && a.epi != EPI_STORE_F32) return -2;
    if (partial && (a.bias != nullptr || a.act != ACT_NONE)) return -2;
    if (a.N % 64 != 0 || a.K % 64 != 0 || a.lda % 4 != 0 || a.ldc % 4 != 0) return -2;
    if (a.ksplit != (partial ? gemm_partial_splits(a.M, a.N, a.K, false) : 1)) return -2;
    // 24-layer step, 16 x 7 rows: 64 x 64 tiles 5.4 ms, 64 x 32 4.0 (128 workgroups for ff linear1 become
    // 256); 16 x 14: 6.1 and 6.2
    if (a.M <= 16) return launch_f32_tile<1, 1>(a, st);
    if (a.M <= 32) return launch_f32_tile<2, 1>(a, st);
    if (a.M <= 64) return launch_f32_tile<4, 1>(a, st);
    if (a.M <= 192) return launch_f32_tile<4, 2>(a, st);
    return launch_f32_tile<4, 4>(a, st);
}

// ---------------------------------------------------------------- launch

template <int MT, int WK, int NT, int EPI, int ACT, bool BIAS = false>
static int launch_reg(GemmArgs a, int ksplit, hipStream_t st) {
    if (a.N % (16 * NT) != 0 || ksplit < 1 || a.K % (64 * ksplit) != 0 || a.K / (64 * ksplit) < WK) return -2;
    if (ksplit > 1 && EPI != EPI_PARTIAL) return -2;
    if (EPI == EPI_STORE_FRAG && a.N % 64 != 0) return -2;
    a.ksplit = ksplit;
    const int tiles = (a.N / (16 * NT)) * ((a.M + 16 * MT - 1) / (16 * MT)) * ksplit;
    hipLaunchKernelGGL((gemm_bf16_kernel<MT, WK, EPI, ACT, NT, BIAS>), dim3(tiles), dim3(64 * WK), 0, st, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int MT, int NT, int NW, int EPI, int ACT, bool BIAS>
static int launch_panel(GemmArgs a, int ksplit, hipStream_t st) {
    if (a.N % (16 * NT * NW) != 0 || ksplit < 1 || a.K % (128 * ksplit) != 0 || a.ldc % 4 != 0) return -2;
    if (ksplit > 1 && EPI != EPI_PARTIAL) return -2;
    a.ksplit = ksplit;
    const int tiles = (a.N / (16 * NT * NW)) * ((a.M + 16 * MT - 1) / (16 * MT)) * ksplit;
    hipLaunchKernelGGL((gemm_panel_kernel<MT, NT, NW, EPI, ACT, BIAS>), dim3(tiles), dim3(64 * NW), 0, st, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

static int device_cus() {
    static int cus = 0;
    if (cus == 0) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0)
            cus = n;
        else
            cus = 256;
    }
    return cus;
}

// The kernel, tile and K splits of one 16-bit GEMM.
enum Gemm16 : int {
    REG_64x64,          // gemm_bf16_kernel<4, 4, .., 4>: 4 waves split K
    REG_64x32,          // gemm_bf16_kernel<4, 4, .., 2>: 4 waves split K
    PANEL_64x128,       // gemm_panel_kernel<4, 2, 4>
    PANEL_128x128,      // gemm_panel_kernel<8, 2, 4>
    PANEL_112x256,      // gemm_panel_kernel<7, 4, 4>
    REG_128x16,         // gemm_bf16_kernel<8, 2, .., 1>: any N % 16 == 0, K % 128 == 0
    REG_FEW,            // at most 128 rows: the shapes of launch_few
};
struct Plan16 { Gemm16 kind; int ks; };

// Few rows: the waves of a workgroup split K.  Many rows: the tile that fills the CUs.  Between them
// no tile is best for long (a workgroup more on some CU costs a whole round of K steps), so the
// choice is a model of each kernel's time,
//   t = t0 + steps (p + q load) + r load  [us],  load = most workgroups on a CU, steps = 32-deep K steps,
// fitted to its times at the encoder's seven shapes (N 256-4,096, K 256-4,352) over 130-57,344 rows
// with weights from HBM; the model's choice is on average 1.5 % slower than the best of the five.
// The K slabs of a residual projection cost the LayerNorm that adds them, and the stores, about
// 1.2 us per slab per 1,000 x 1,024 outputs.
// Measured against what these rows had (128 x 16 register tiles below 2,048 rows, 128/224/256-row
// tiles with both operands in LDS above), us per launch, random data:
//   rows                        256          640          1,024        2,048        3,584
//   ff linear1 (4,096 x 1,024)  11.2 -> 7.9  19.5 -> 12.7 27.7 -> 13.3 21.6 -> 21.0 35.4 -> 30.9
//   ff linear2 (1,024 x 4,096)  10.8 -> 7.5  25.1 -> 14.7 50.8 -> 15.5 26.1 -> 23.5 36.5 -> 33.8
//   q/k/v (3,072 x 1,024)        9.3 -> 7.0  14.5 ->  9.3 22.9 -> 12.4 21.0 -> 18.8 30.5 -> 28.2
//   linear_out (1,024 x 1,024)   4.9 -> 4.0   8.1 ->  6.0 11.0 ->  6.5 12.0 ->  8.7 15.1 -> 13.6
static Plan16 plan16(int M, int N, int K, int epi) {
    const bool partial = epi == EPI_PARTIAL;
    if (M <= 128) return Plan16{REG_FEW, !partial ? 1 : K == 1024 && N % 32 == 0 ? 2 : K % (128 * KSPLIT) == 0 ? KSPLIT : 1};
    struct Model { Gemm16 kind; int rows, cols, waves_k; double t0, p, q, r; };
    static const Model models[] = {
        {REG_64x64, 64, 64, 4, 0.0, 0.0137, 0.0915, 3.151},
        {REG_64x32, 64, 32, 4, 0.98, 0.0160, 0.0690, 0.752},
        {PANEL_64x128, 64, 128, 0, 1.05, 0.0926, 0.0925, 1.867},
        {PANEL_128x128, 128, 128, 0, 0.90, 0.1222, 0.1117, 3.915},
        {PANEL_112x256, 112, 256, 0, 0.28, 0.1726, 0.1656, 6.654},
    };
    const long cus = device_cus();
    Plan16 best{REG_128x16, partial && K % (128 * KSPLIT) == 0 ? KSPLIT : 1};
    double best_t = 1e300;
    for (const Model& m : models)
        for (int ks = 1; ks <= (partial ? KSPLIT : 1); ks *= 2) {
            // the panel kernel runs whole groups of four K steps; a register wave needs a 64-deep chunk
            if (N % m.cols != 0 || K % (128 * ks) != 0 || (ks > 1 && K / ks < 256) || K / (64 * ks) < m.waves_k) continue;
            const long load = ((long)(N / m.cols) * ((M + m.rows - 1) / m.rows) * ks + cus - 1) / cus;
            double t = m.t0 + K / (32.0 * ks) * (m.p + m.q * load) + m.r * load;
            if (partial) t += 1.2 * ks * ((double)M * N / 1024e3);
            if (t < best_t) { best_t = t; best = Plan16{m.kind, ks}; }
        }
    return best;
}

int gemm_partial_splits(int M, int N, int K, bool half_data) {
    if (half_data) return plan16(M, N, K, EPI_PARTIAL).ks;
    // fp32: by K alone (see gemm_f32_kernel), at least a 64-wide chunk for each wave where it can be had
    return K % 256 == 0 && K >= 2048 ? KSPLIT : K % 128 == 0 && K >= 1024 ? 2 : 1;
}

// At most 128 rows: the smallest tile (16 x 16, 16 x 32, 32 x 32, 64 x 32) that gives no CU a second
// workgroup.  Such a launch streams its 2-8 MB of weights once, whatever the tile, so what counts is
// that every CU has part of them in flight; a wider tile only cuts the re-reads of the activation
// rows.  Four waves split K, eight where the K range is long (the subsampling's out: 4,352) and in the
// tallest tile.  us per launch, weights from HBM, against the tiles tuned at 128 rows that all of these
// had (32 x 64, 64 x 32, 32 x 32, all with 8 waves):
//   rows                                    2             16            32            64            128
//   ff linear1 (4,096 x 1,024)              6.1 -> 4.0    6.1 -> 4.0    6.1 -> 4.4    5.9 -> 4.8    5.8
//   ff linear2 (1,024 x 4,096, 4 splits)    5.4 -> 3.8    5.4 -> 4.0    5.4 -> 4.3    5.4 -> 4.8    5.9
//   q/k/v (3,072 x 1,024)                   5.7 -> 3.6    5.7 -> 3.7    5.7 -> 4.0    5.7 -> 4.5    5.5
//   pointwise_conv1 (2,048 x 1,024, GLU)    4.0 -> 3.5    4.2 -> 3.9    4.4 -> 3.8    4.3 -> 3.8    4.3 -> 4.2
//   linear_out (1,024 x 1,024, 2 splits)    2.9 -> 2.7    3.0 -> 2.7    3.0 -> 2.8    3.1 -> 3.0    3.4 -> 3.2
//   subsampling out (1,024 x 4,352)         8.0 -> 7.2    8.4 -> 7.5    9.4 -> 7.2    9.0 -> 7.1    8.7
template <int EPI, int ACT, bool BIAS, int MT, int NT>
static int launch_few_tile(const GemmArgs& a, int ks, hipStream_t st) {
    if (a.K / (64 * ks) >= 8 && (a.K / ks >= 2048 || MT == 4)) return launch_reg<MT, 8, NT, EPI, ACT, BIAS>(a, ks, st);
    return launch_reg<MT, 4, NT, EPI, ACT, BIAS>(a, ks, st);
}
template <int EPI, int ACT, bool BIAS>
static int launch_few(const GemmArgs& a, int ks, hipStream_t st) {
    const int cus = device_cus();
    auto fits = [&](int mt, int nt) { return a.N / (16 * nt) * ((a.M + 16 * mt - 1) / (16 * mt)) * ks <= cus; };
    if (a.K / (64 * ks) >= 4) {
        if constexpr (EPI != EPI_GLU)
            if (fits(1, 1)) return launch_few_tile<EPI, ACT, BIAS, 1, 1>(a, ks, st);
        if (a.N % 32 == 0) {
            if (fits(1, 2)) return launch_few_tile<EPI, ACT, BIAS, 1, 2>(a, ks, st);
            if (fits(2, 2)) return launch_few_tile<EPI, ACT, BIAS, 2, 2>(a, ks, st);
            return launch_few_tile<EPI, ACT, BIAS, 4, 2>(a, ks, st);
        }
    }
    return launch_reg<8, 2, EPI == EPI_GLU ? 2 : 1, EPI, ACT, BIAS>(a, ks, st);
}

template <int EPI, int ACT, bool BIAS>
static int launch_16(const GemmArgs& a, int ks, hipStream_t st) {
    const Plan16 p = plan16(a.M, a.N, a.K, EPI);
    if (p.ks != ks) return -2;              // EPI_PARTIAL: the caller sized its slabs by another plan
    switch (p.kind) {
        case REG_64x64: return launch_reg<4, 4, 4, EPI, ACT, BIAS>(a, ks, st);
        case REG_64x32: return launch_reg<4, 4, 2, EPI, ACT, BIAS>(a, ks, st);
        case PANEL_64x128: return launch_panel<4, 2, 4, EPI, ACT, BIAS>(a, ks, st);
        case PANEL_128x128: return launch_panel<8, 2, 4, EPI, ACT, BIAS>(a, ks, st);
        case PANEL_112x256: return launch_panel<7, 4, 4, EPI, ACT, BIAS>(a, ks, st);
        case REG_FEW: return launch_few<EPI, ACT, BIAS>(a, ks, st);
        default: return launch_reg<8, 2, EPI == EPI_GLU ? 2 : 1, EPI, ACT, BIAS>(a, ks, st);
    }
}

template <int EPI, bool BIAS>
static int launch_act(const GemmArgs& a, hipStream_t st) {
    switch (a.act) {
        case ACT_NONE: return launch_16<EPI, ACT_NONE, BIAS>(a, 1, st);
        case ACT_SILU: return BIAS ? -2 : launch_16<EPI, ACT_SILU, false>(a, 1, st);
        case ACT_RELU: return launch_16<EPI, ACT_RELU, BIAS>(a, 1, st);
        default: return -2;
    }
}

// The encoder's projections have no bias; the subsampling front-end's GEMMs have one (a template
// parameter: a runtime-optional bias in the encoder's own GEMMs made their epilogues larger and cost
// ~2 us per launch at 128 rows).
static int launch_half(const GemmArgs& a, hipStream_t st) {
    const bool bias = a.bias != nullptr;
    switch (a.epi) {
        case EPI_STORE: return bias ? launch_act<EPI_STORE, true>(a, st) : launch_act<EPI_STORE, false>(a, st);
        case EPI_STORE_F32: return bias ? launch_act<EPI_STORE_F32, true>(a, st) : launch_act<EPI_STORE_F32, false>(a, st);
        case EPI_SUBFLAT: return bias ? launch_act<EPI_SUBFLAT, true>(a, st) : -2;
        default: break;
    }
    if (bias) return -2;
    switch (a.epi) {
        case EPI_STORE_FRAG: return a.N % 64 == 0 ? launch_act<EPI_STORE_FRAG, false>(a, st) : -2;
        case EPI_QKV_RING: return launch_16<EPI_QKV_RING, ACT_NONE, false>(a, 1, st);
        case EPI_GLU: return launch_16<EPI_GLU, ACT_NONE, false>(a, 1, st);
        case EPI_PARTIAL: return a.act == ACT_NONE ? launch_16<EPI_PARTIAL, ACT_NONE, false>(a, a.ksplit, st) : -2;
        default: return -2;
    }
}

int launch_gemm(const GemmArgs& a, bool half_data, hipStream_t st) {
    if (a.M <= 0 || a.N <= 0 || a.K <= 0) return -2;
    // GLU pairs: 16-bit only, no activation, whole 32-column value/gate blocks, half the columns out
    if (a.epi == EPI_GLU && (!half_data || a.act != ACT_NONE || a.bias || a.N % 32 != 0 || a.ldc < a.N / 2 || a.ldc % 4))
        return -2;
    if (a.epi == EPI_QKV_RING) {
        // 16-bit only, no activation; the rows are whole streams of T frames; every ring row written
        // is outside the step's window (L + T <= R)
        const QkvRing& r = a.ring;
        if (!half_data || a.act != ACT_NONE || a.bias || !r.kring || !r.vring || !r.rows || r.T < 1 || r.H < 1 ||
            a.N != 3 * r.H * 128 || a.M % r.T != 0 || r.L + r.T > r.R || a.ldc < r.H * 128)
            return -2;
    }
    if (!half_data) return launch_f32(a, st);
    if (a.K % 128 != 0) return -2;
    if (a.epi == EPI_SUBFLAT) {
        const SubFlat& f = a.flat;
        if (!f.vlen || f.T3 < 1 || f.F3 < 1 || f.drop < 0 || f.T != f.T3 - f.drop || a.M % (f.T3 * f.F3) != 0 ||
            (f.F3 * a.N) % 64)
            return -2;
    }
    return launch_half(a, st);
}

}  // namespace ud
