// All layers of one step of a few sequences in ONE launch.
//
// A batched step through kernels_gemm.h and kernels_attn.h is five dependent launches per layer,
// each 4 to 7 us of which the weights are 0.3 to 1.6: start, arguments, one trip to memory for the
// operands, products, merge, end.  Here one workgroup per compute unit stays for the whole step and
// the phases of a layer
//   norm1 + QKV -> attention -> W_o + residual -> norm2 + FFN1 -> FFN2 + residual
// hand their rows on through cells, 8-byte {value, tag} pairs as in kernels_persist.h: written with
// one device-scope store, polled with device-scope loads until the tag is the one expected.  A phase's
// weights, norm parameters and cached keys and values are requested before its inputs are polled.
//
// The arithmetic is that of the launches, bit for bit: a projection is gemm16_kernel's 16 x 16 tile (K
// over eight wavefronts, the same products in the same order, partial sums added in order), the
// attention attn_decode64_kernel's, the LayerNorm layernorm_rows_kernel's.  So which of the two
// forms runs a step is a matter of speed alone.  (src/transformer/inference.cpp:184-249)
//
// What bounds it: five hand-offs per layer, and between them chains of a few hundred instructions on eight wavefronts.
// From the last store of a phase to the rows of the next being there / from there to its last store, us, one layer of the
// Llama block d768, 4 sequences behind 64 positions: QKV 1.1 / 1.8, attention 0.6 / 1.8, W_o 1.8 / 1.1, FFN1 1.2 / 2.8,
// FFN2 2.2 / 1.6 (0.9 of it products, 16-row tiles for 4 rows; 128 KB of weights through one compute unit), 16.1 in
// all; 16 sequences behind 200 1.4 / 2.1, 0.9 / 2.8, 2.3 / 1.6, 1.7 / 3.1, 1.7 / 3.7, 21.3.  The matrix cores are busy
// 8 % of the time at 4 sequences, and the 251 MB that miss the L2s (226 of them weights) go at 1.9 TB/s.  Per step,
// launches -> this, behind 184 positions: Llama block 2 sequences 249 us -> 144, 4 257 -> 158, 8 276 -> 173, 16 318 -> 193;
// GPT-2 block d768 2 sequences 289 -> 166, 16 353 -> 222; Llama block, 16 sequences behind 1884 positions 523 -> 444:
// 188 MB of cache per layer in the 33 us of its 53 that the attention takes.
// Built for the d512 and d768 shapes.  d1024 / F4096 would fit (64 + 192 workgroups, two FFN1 tiles each) and is
// launches, 337 us at 2 sequences and 403 at 16 behind 128: not tried.  So are more than 16 sequences (Llama, behind
// 128: 16 188, 17 324), which need a second tile of rows per product.
//
// The order things are sent in is most of the design.  A wavefront's loads return in the order they
// went out, and a workgroup's stores leave behind what its other wavefronts have asked for: weights are
// requested one phase ahead and not two, and nobody requests anything between a phase's barrier and its
// stores (without the barrier behind the stores a layer took 19.5 us instead of 16.8).
#pragma once

#include "kernels_attn.h"
#include "kernels_gemm.h"
#include "kernels_persist.h"

namespace gh {

constexpr int kResidentThreads = 512, kResidentGrid = 256, kResidentRows = 16;
constexpr int kResidentTableBytes = 16384;                // page tables of all sequences, in LDS
constexpr int kResidentRounds = 4;
constexpr int kResidentItems = 2 * kResidentGrid * kResidentRounds;  // (sequence, head, run of positions) of the attention: two per workgroup and round

struct ResidentCtl {
    unsigned abort;  // set by any workgroup that gave up waiting
    unsigned where;  // the tag it was waiting for (diagnostics)
};

struct ResidentParams {
    const float* layer0;  // the layers' tensors, as layer_at() says
    const float *rope_cos, *rope_sin;
    float* x;  // [B][D] residual rows: in and out
    KvLayout kv;
    Cell* cells;  // resident_cells() of them
    ResidentCtl* ctl;
    int B, L;
    int pos;        // positions already in the cache
    int chunk;      // positions per item of the attention
    unsigned epoch;  // tags are (epoch + layer) * 8 + phase + 1
    unsigned spin_limit;
};

// Cells of x behind a layer and behind its attention half [D][B] each, q, new keys and values [B][D], attention
// output [D][B], hidden [F][B], and the items' shares of a longer context [items][66].
__host__ __device__ constexpr size_t resident_cells(size_t D, size_t F, size_t B) {
    return (6 * D + F) * B + static_cast<size_t>(kResidentItems) * 66;
}

// Where operand rows lie: two columns of all rows follow each other, so that a load of 16 bytes per lane, two
// columns of a row with their tags, reads whole lines.  (A row's 16 columns in one line, which suits
// the wavefronts that write them: 8 sequences 166 -> 189 us per step, 4 152 -> 155.)
__device__ __forceinline__ int operand_cell(int k, int r, int rows) {
    return ((((k >> 4) * 2 + ((k >> 1) & 1)) * 4 + ((k >> 2) & 3)) * rows + r) * 2 + (k & 1);
}

// RP: rows a load of operands is dealt for (B <= RP, of 4, 8 and 16).  A product takes row lane % 16, so with few
// rows most lanes would have nothing to load: 16 / RP units of two columns share a load instead, and
// move to their lanes inside the registers.
// ROUNDS: more items of the attention than halves of workgroups.  A variant of its own: the loop over
// rounds costs a step that has only one 1 to 3 %.  (A wavefront's next 32 positions requested before the
// present ones are worked on: spills at d768, 2 to 6 % slower at every context but one.)
template <int KD, int KF, bool MODERN, int RP, bool ROUNDS>
__global__ __launch_bounds__(kResidentThreads) void resident_layers_kernel(const ResidentParams p) {
    constexpr int D = KD * 256, F = KF * 256, HS = 64, H = D / HS, KW = 8;
    constexpr int ND = D / KW / 16, NF = F / KW / 16;  // 16-column blocks of a wavefront's share of K
    constexpr int TO = D / 16, TQ = 3 * D / 16, T1 = (MODERN ? 2 * F : F) / 16;
    constexpr int G = kResidentGrid, NO = G - TO;
    constexpr int LDX = D + 4;
    static_assert(TO + TQ <= G && T1 <= 2 * NO, "every phase in one round");
    static_assert(TO % 8 == 0 && TQ % 8 == 0 && G % 8 == 0, "an item's XCD is its number modulo 8");
    __shared__ float red[2][2][KW][256];  // [phase parity][tile][wavefront][row * 16 + column]
    __shared__ float ssq[2][KW][16];
    __shared__ float part[2][2][4][68];  // [parity of the round][half]: as in attn_decode64_kernel
    __shared__ float held[ROUNDS ? kResidentRounds : 1][2][66];  // the first run of a context in several
    __shared__ float rows[MODERN ? 1 : kResidentRows * LDX];
    __shared__ float mean[16], scale[16];
    extern __shared__ int ptab[];  // [B][pages_per_seq]
    int tid = threadIdx.x;
    const int wg = blockIdx.x, B = p.B, pos = p.pos;
    int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // (a step behind one that gave up has nothing to work on)
    if (tid == 0) g_wait_abandoned = __hip_atomic_load(&p.ctl->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int i = tid; i < B * p.kv.pages_per_seq; i += kResidentThreads) ptab[i] = p.kv.page_table[i];
    __syncthreads();
    if (g_wait_abandoned) return;

    const bool owner = wg < TO;             // 16 columns of the residual rows: W_o and FFN2
    const bool has_qkv = wg >= TO && wg < TO + TQ;
    const int u1 = wg - TO;                 // tiles u1 and u1 + NO of FFN1
    // Attention items: first to the workgroups that have nothing to do beside QKV, the owners last.
    const int order = wg >= TO + TQ ? wg - (TO + TQ) : wg >= TO ? wg - TO + (G - TO - TQ) : wg + (G - TO);
    const int ctx = pos + 1, nchunk = (ctx + p.chunk - 1) / p.chunk;
    const int items = B * H * nchunk;
    const int rounds = ROUNDS ? (items + 2 * G - 1) / (2 * G) : 1;
    const bool has_items = order < items;

    const __amdgpu_buffer_rsrc_t rs = make_buffer(p.cells, static_cast<unsigned>(resident_cells(D, F, B) * sizeof(Cell)));
    const int c_x = 0, c_mid = D * B, c_q = 2 * D * B, c_at = 5 * D * B, c_hid = 6 * D * B, c_part = (6 * D + F) * B;
    constexpr unsigned kPastEnd = 0x80000000u;

    // the thread's pair of outputs in a tile: row ei, columns ej and ej + 1
    const bool e_live = tid < 8 * B;
    const int ei = tid >> 3, ej = (tid & 7) * 2;

    const auto give_up = [&](unsigned tag) {
        __hip_atomic_store(&p.ctl->where, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&p.ctl->abort, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        g_wait_abandoned = 1u;
    };
    // one more look without success: is it time to stop waiting?
    const auto hopeless = [&](unsigned& spins) {
        ++spins;
        return spins > p.spin_limit
               || ((spins & 63u) == 0u && __hip_atomic_load(&p.ctl->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u);
    };

    float r0 = 0.0f, r1 = 0.0f;  // the owner thread's pair of the residual rows
    if (owner && e_live) {
        r0 = p.x[static_cast<size_t>(ei) * D + wg * 16 + ej];
        r1 = p.x[static_cast<size_t>(ei) * D + wg * 16 + ej + 1];
    }

    for (int l = 0; l < p.L; l++) {
        const LayerPtrs w = layer_at<KD, KF, MODERN>(p.layer0, l);
        asm volatile("" : "+v"(tid));  // addresses are formed per layer, not kept across the loop
        wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        lane = tid & 63;
        const int j = lane & 15, g = lane >> 4;
        const int fr = lane >> 2, fc = lane & 3;
        const int from_lane = (j * 4 + g) * 4;
        const unsigned sb = (p.epoch + static_cast<unsigned>(l)) * 8u;
        const auto to_operand = [&](const float4& v) {
            return make_float4(__int_as_float(__builtin_amdgcn_ds_bpermute(from_lane, __float_as_int(v.x))),
                               __int_as_float(__builtin_amdgcn_ds_bpermute(from_lane, __float_as_int(v.y))),
                               __int_as_float(__builtin_amdgcn_ds_bpermute(from_lane, __float_as_int(v.z))),
                               __int_as_float(__builtin_amdgcn_ds_bpermute(from_lane, __float_as_int(v.w))));
        };
        // NB blocks of rows n0 .. + 15 of a matrix of K columns: this wavefront's share of K from block b0 on
        const auto fetch_rows = [&](const float* W, int K, int n0, int k0, auto& out) {
            const float* at = W + static_cast<size_t>(n0 + fr) * K + k0 + fc * 4;
#pragma unroll
            for (int i = 0; i < static_cast<int>(sizeof(out) / sizeof(float4)); i++) out[i] = *reinterpret_cast<const float4*>(at + 16 * i);
        };
        const auto to_operands = [&](auto& v) {
#pragma unroll
            for (int i = 0; i < static_cast<int>(sizeof(v) / sizeof(float4)); i++) v[i] = to_operand(v[i]);
        };
        // Waits for columns k0 .. of the operand rows in the cells from `first` on.
        const auto poll_rows = [&](int first, int k0, unsigned tag, auto& a) {
            constexpr int N = sizeof(a) / sizeof(float4);
            constexpr int PACK = 16 / RP, LOADS = 2 * N / PACK;  // units of a lane group per load
            const int r = j % RP, q = j / RP;                    // unit 2 * block + half = PACK * i + q
            const unsigned line = static_cast<unsigned>(B) * 128u;  // bytes of a 16-column block
            unsigned at = static_cast<unsigned>(first) * 8u + static_cast<unsigned>(k0 >> 4) * line;
            at += static_cast<unsigned>(((q & 1) * 4 + g) * B + r) * 16u + static_cast<unsigned>(q >> 1) * line;
            if (r >= B) at = kPastEnd;
            unsigned spins = 0;
            v4i u[LOADS];
            if constexpr (LOADS > 6 && RP < 16) {
                // the last of the loads alone until its columns are there
                for (;;) {
                    const v4i w = coherent_load16(rs, at + (PACK == 1 ? (LOADS - 1) * (line / 2) : (PACK * (LOADS - 1) >> 1) * line));
                    if (__all((w.y == static_cast<int>(tag) && w.w == static_cast<int>(tag)) || r >= B)) break;
                    if (hopeless(spins)) {
                        give_up(tag);
                        break;
                    }
                }
            }
            for (;;) {
#pragma unroll
                for (int i = 0; i < LOADS; i++)
                    u[i] = coherent_load16(rs, at + (PACK == 1 ? i * (line / 2) : (PACK * i >> 1) * line));
                bool ok = true;
#pragma unroll
                for (int i = 0; i < LOADS; i++) ok = ok && u[i].y == static_cast<int>(tag) && u[i].w == static_cast<int>(tag);
                if (__all(ok || r >= B)) break;
                if (hopeless(spins)) {
                    give_up(tag);
                    break;
                }
            }
#pragma unroll
            for (int i = 0; i < N; i++) {
                float v[4];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const v4i& w = u[(2 * i + h) / PACK];
                    const float x = __int_as_float(w.x), y = __int_as_float(w.z);
                    const int from = (2 * i + h) % PACK;  // lanes RP * from .. of 16 hold it
                    v[2 * h] = from == 0 ? x : from == 1 ? dpp_move<0x100 + (RP == 8 ? 8 : 4), 0xF>(x, 0.0f)
                               : from == 2               ? dpp_move<0x108, 0xF>(x, 0.0f) : dpp_move<0x10C, 0xF>(x, 0.0f);
                    v[2 * h + 1] = from == 0 ? y : from == 1 ? dpp_move<0x100 + (RP == 8 ? 8 : 4), 0xF>(y, 0.0f)
                                   : from == 2               ? dpp_move<0x108, 0xF>(y, 0.0f) : dpp_move<0x10C, 0xF>(y, 0.0f);
                }
                a[i] = make_float4(v[0], v[1], v[2], v[3]);
            }
        };
        const auto multiply = [&](const auto& a, const auto& b, v4f& acc) {
#pragma unroll
            for (int i = 0; i < static_cast<int>(sizeof(a) / sizeof(float4)); i++) {
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].x, b[i].x, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].y, b[i].y, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].z, b[i].z, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].w, b[i].w, acc, 0, 0, 0);
            }
        };
        const auto leave = [&](int parity, int tile, const v4f& acc) {
#pragma unroll
            for (int r = 0; r < 4; r++) red[parity][tile][wave][(4 * g + r) * 16 + j] = acc[r];
        };
        const auto sum_pair = [&](int parity, int tile, float& v0, float& v1) {
            v0 = v1 = 0.0f;
#pragma unroll
            for (int q = 0; q < KW; q++) {
                const float2 v = *reinterpret_cast<const float2*>(&red[parity][tile][q][ei * 16 + ej]);
                v0 += v.x;
                v1 += v.y;
            }
        };
        // The norm of the rows polled.  RMSNorm: the gain, and the wavefront's share of the sums of
        // squares for rms() behind the barrier.  LayerNorm: whole rows through LDS (two barriers).
        const auto norm_rows = [&](float4 (&a)[ND], const float4 (&gain)[ND], const float4 (&shift)[ND], int parity) {
            if constexpr (MODERN) {
                float ss = 0.0f;
#pragma unroll
                for (int i = 0; i < ND; i++) {
                    ss += fmaf(a[i].w, a[i].w, fmaf(a[i].z, a[i].z, fmaf(a[i].x, a[i].x, a[i].y * a[i].y)));
                    a[i] = make_float4(a[i].x * gain[i].x, a[i].y * gain[i].y, a[i].z * gain[i].z, a[i].w * gain[i].w);
                }
                ss += __shfl_xor(ss, 16, kWave);
                ss += __shfl_xor(ss, 32, kWave);
                if (lane < 16) ssq[parity][wave][lane] = ss;
            } else {
#pragma unroll
                for (int i = 0; i < ND; i++)
                    if (j < B) *reinterpret_cast<float4*>(&rows[j * LDX + wave * (D / KW) + 16 * i + 4 * g]) = a[i];
                __syncthreads();
                for (int r = wave; r < B; r += KW) {
                    float v[D / 64];
                    float width = D;
                    asm volatile("" : "+v"(width));
                    float s = 0.0f;
#pragma unroll
                    for (int i = 0; i < D / 64; i++) {
                        v[i] = rows[r * LDX + 64 * i + lane];
                        s += v[i];
                    }
                    const float mu = wave_sum(s) / width;
                    float var = 0.0f;
#pragma unroll
                    for (int i = 0; i < D / 64; i++) var = fmaf(v[i] - mu, v[i] - mu, var);
                    const float inv_std = 1.0f / sqrtf(wave_sum(var) / width + kNormEps);
                    if (lane == 0) {
                        mean[r] = mu;
                        scale[r] = inv_std;
                    }
                }
                __syncthreads();
                const float mu = mean[j], inv_std = scale[j];
#pragma unroll
                for (int i = 0; i < ND; i++)
                    a[i] = make_float4(fmaf(inv_std, gain[i].x * (a[i].x - mu), shift[i].x),
                                       fmaf(inv_std, gain[i].y * (a[i].y - mu), shift[i].y),
                                       fmaf(inv_std, gain[i].z * (a[i].z - mu), shift[i].z),
                                       fmaf(inv_std, gain[i].w * (a[i].w - mu), shift[i].w));
            }
        };
        const auto fetch_norm = [&](const float* gamma, const float* beta, float4 (&gain)[ND], float4 (&shift)[ND]) {
            const int at = wave * (D / KW) + 4 * g;
#pragma unroll
            for (int i = 0; i < ND; i++) {
                gain[i] = *reinterpret_cast<const float4*>(gamma + at + 16 * i);
                if constexpr (!MODERN) shift[i] = *reinterpret_cast<const float4*>(beta + at + 16 * i);
                else shift[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
        };
        const auto rms = [&](int parity) {
            float ms = 0.0f;
#pragma unroll
            for (int q = 0; q < KW; q++) ms += ssq[parity][q][ei];
            return 1.0f / sqrtf(ms / static_cast<float>(D) + kNormEps);
        };

        // ===== norm1 + QKV
        if (has_qkv) {
            float4 b[ND], a[ND], gain[ND], shift[ND];
            const int n0 = u1 * 16, n = n0 + ej;
            fetch_rows(w.wqkv, D, n0, wave * (D / KW), b);
            fetch_norm(w.g1, w.be1, gain, shift);
            float b0 = 0.0f, b1 = 0.0f, cs = 1.0f, sn = 0.0f;
            if (e_live) {
                b0 = w.bqkv[n];
                b1 = w.bqkv[n + 1];
                if (MODERN && n < 2 * D) {
                    const int jj = ((n % D) % HS) >> 1;
                    cs = p.rope_cos[pos * (HS / 2) + jj];
                    sn = p.rope_sin[pos * (HS / 2) + jj];
                }
            }
            if (l == 0) {
                const float* xr = p.x + static_cast<size_t>(min(j, B - 1)) * D + wave * (D / KW) + 4 * g;
#pragma unroll
                for (int i = 0; i < ND; i++) a[i] = *reinterpret_cast<const float4*>(xr + 16 * i);
                to_operands(b);
            } else {
                to_operands(b);
                poll_rows(c_x, wave * (D / KW), sb - 8u + 5u, a);
            }
            norm_rows(a, gain, shift, 0);
            v4f acc = {0.f, 0.f, 0.f, 0.f};
            multiply(a, b, acc);
            leave(0, 0, acc);
            __syncthreads();
            if (e_live) {
                float v0, v1;
                sum_pair(0, 0, v0, v1);
                if (MODERN) {
                    const float r = rms(0);
                    v0 *= r;
                    v1 *= r;
                }
                float x0 = v0 + b0, x1 = v1 + b1;
                if (MODERN && n < 2 * D) {
                    const float ra = x0 * cs - x1 * sn;
                    const float rc = x0 * sn + x1 * cs;
                    x0 = ra;
                    x1 = rc;
                }
                const int sec = n / D, c = n - sec * D;
                cell_put2(rs, c_q + sec * D * B + ei * D + c, x0, x1, sb + 1u);
                if (sec > 0) {
                    const int page = ptab[ei * p.kv.pages_per_seq + (pos >> p.kv.page_shift)];
                    const int slot = pos & ((1 << p.kv.page_shift) - 1);
                    const size_t run = ((static_cast<size_t>(l) * p.kv.n_pages + page) * 2 + (sec - 1)) * H + (c >> 6);
                    *reinterpret_cast<float2*>(p.kv.pool + ((run << p.kv.page_shift) + slot) * HS + (c & 63)) = make_float2(x0, x1);
                }
            }
            __syncthreads();  // nobody's loads go out in front of these stores
        }

        // ===== attention: attn_decode64_kernel's workgroup is half of this one.  With more items than halves of
        // workgroups they go in rounds, and the runs of a longer context are folded when every round's are out (a run in
        // a later round may be what another workgroup's fold waits for).
        if (has_items) {
            const int half = wave >> 2, wv = wave & 3;
            const int sub = lane >> 4, dl = lane & 15;
            const int shift = p.kv.page_shift;
            const size_t head_stride = static_cast<size_t>(HS) << shift, kv_stride = head_stride * H;
            const float* pool = p.kv.pool + static_cast<size_t>(l) * p.kv.n_pages * 2 * kv_stride;
            const auto publish = [&](int seq, int h, float v) {  // two columns per store
                const float next = dpp_move<0xB1, 0xF>(v, 0.0f);
                if (!(lane & 1)) cell_put2(rs, c_at + operand_cell(h * HS + lane, seq, B), v, next, sb + 2u);
            };
            // the other runs of a context whose first gave M, L and o, folded in order (attn_merge)
            const auto fold = [&](int item, float M, float L, float o) {
                const int pair = item / nchunk, seq = pair / H, h = pair - seq * H;
                float all = M;
                float cm = 0.0f, cl = 0.0f, co = 0.0f;
                const auto look = [&](int c) {
                    const Cell* theirs = p.cells + c_part + (item + c) * 66;
                    unsigned spins = 0;
                    for (;;) {
                        const bool got_m = cell_get(theirs, sb + 6u, cm);
                        const bool got_l = cell_get(theirs + 1, sb + 6u, cl);
                        const bool got_o = cell_get(theirs + 2 + lane, sb + 6u, co);
                        if (__all(got_m && got_l && got_o)) break;
                        if (hopeless(spins)) {
                            give_up(sb + 6u);
                            break;
                        }
                    }
                };
                for (int c = 1; c < nchunk; c++) {
                    look(c);
                    all = fmaxf(all, cm);
                }
                float f = expf(M - all);
                float Ls = 0.0f, os = 0.0f;
                Ls += L * f;
                os += o * f;
                for (int c = 1; c < nchunk; c++) {
                    look(c);
                    f = expf(cm - all);
                    Ls += cl * f;
                    os += co * f;
                }
                publish(seq, h, os * (1.0f / Ls));
            };
            // this wavefront's positions [t0, t1) of an item, and where its rows are
            const auto run_of = [&](int item, int& seq, int& h, int& ck, int& t0, int& t1) {
                const int pair = item / nchunk;
                ck = item - pair * nchunk;
                seq = pair / H;
                h = pair - seq * H;
                const int p0 = ck * p.chunk, p1 = min(ctx, p0 + p.chunk);
                const int run = ((((p1 - p0) + 3) / 4) + 31) & ~31;
                t0 = p0 + wv * run;
                t1 = min(p1, t0 + run);
            };
            // Brings rows [from, t1) of a run into this XCD's L2: lane i its 128-byte line of 64.
            const auto touch = [&](int seq, int h, int from, int t1) {
                float v = 0.0f;
                for (int tb = from; tb < t1; tb += 32) {
                    const float* at = pool + h * head_stride + static_cast<size_t>(ptab[seq * p.kv.pages_per_seq + (tb >> shift)]) * 2 * kv_stride
                                      + static_cast<size_t>(tb & ((1 << shift) - 1)) * HS + lane * 32;
                    if (tb + (lane >> 1) < min(t1, pos)) v += at[0] + at[kv_stride];
                }
                return v;
            };
            // Rows that come from beyond the L2 only when q is there are most of what a context costs.  The
            // workgroups without a tile of QKV have that phase to spare: they touch the rows of their own
            // runs beyond the first 32, and where their second half has no item, it touches those of the
            // workgroups with a tile (an item's XCD is that of its number modulo 8, TO and TQ being multiples
            // of 8).  That pays while all rows of an XCD fit its 4 MB of L2 beside the weights passing through,
            // and from 64 positions on.  us per step, before and after, Llama block: 2 sequences behind 300 159 -> 152,
            // 4 182 -> 170, 8 210 -> 184, 13 226 -> 213; 13 behind 130 198 -> 189; GPT-2 8 behind 300
            // 232 -> 210.  Without the limits: 8 behind 600 238 -> 261, GPT-2 16 behind 30 202 -> 207.
            const bool spare = wg >= TO + TQ;
            constexpr int kTouchPositions = 53248;  // of all heads: 3.25 MB of rows per XCD
            if (spare && half == 1 && order + G >= items && ctx > 64 && B * H * ctx <= kTouchPositions) {
                float touched = 0.0f;
                for (int item = order + (G - TO - TQ); item < min(items, G); item += G - TO - TQ) {
                    int seq, h, ck, t0, t1;
                    run_of(item, seq, h, ck, t0, t1);
                    touched += touch(seq, h, t0, t1);
                }
                asm volatile("" ::"v"(touched));
            }
            for (int round = 0; round < rounds; round++) {
                const int item = order + (2 * round + half) * G;
                const bool live = item < items;
                int seq, h, ck, t0, t1;
                run_of(live ? item : 0, seq, h, ck, t0, t1);
                const int* table = ptab + seq * p.kv.pages_per_seq;
                const float* base = pool + h * head_stride;
                float m = -INFINITY, lsum = 0.0f;
                float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
                if (live && t0 < t1) {
                    float4 k4[8], v4[8];
                    const auto fetch = [&](int tb) {
                        const float* at = base + static_cast<size_t>(table[tb >> shift]) * 2 * kv_stride;
#pragma unroll
                        for (int it = 0; it < 8; it++) {
                            const int tt = tb + it * 4 + sub;
                            k4[it] = make_float4(0.f, 0.f, 0.f, 0.f);
                            v4[it] = make_float4(0.f, 0.f, 0.f, 0.f);
                            if (tt < t1 && tt < pos) {
                                const float* row = at + static_cast<size_t>(tt & ((1 << shift) - 1)) * HS + dl * 4;
                                k4[it] = *reinterpret_cast<const float4*>(row);
                                v4[it] = *reinterpret_cast<const float4*>(row + kv_stride);
                            }
                        }
                    };
                    const bool newest = t1 == ctx;
                    float4 q4, kn, vn;
                    const auto work = [&](int tb) {
                        // The new position goes in ahead of the scores, not between them: only one wavefront of a
                        // head has it (8 sequences behind 300: 211 -> 208 us, 16: 228 -> 225).  Rows without a
                        // condition, by a buffer's end, are 3 us better there and 1 to 2 % worse in rounds.
                        if (pos - tb < 32) {
#pragma unroll
                            for (int it = 0; it < 8; it++)
                                if (it * 4 + sub == pos - tb) {
                                    k4[it] = kn;
                                    v4[it] = vn;
                                }
                        }
                        float sc[8];
#pragma unroll
                        for (int it = 0; it < 8; it++) {
                            const int tt = tb + it * 4 + sub;
                            const float sdot = row16_sum(dot4(q4, k4[it]));
                            sc[it] = tt < t1 ? sdot * 0.125f : -INFINITY;  // 1/sqrt(64)
                        }
                        float mb = sc[0];
#pragma unroll
                        for (int it = 1; it < 8; it++) mb = fmaxf(mb, sc[it]);
                        mb = fmaxf(mb, dpp_move<0x142, 0xA>(mb, mb));
                        mb = fmaxf(mb, dpp_move<0x143, 0xC>(mb, mb));
                        mb = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(mb), 63));
                        const float mn = fmaxf(m, mb);
                        float arg = sc[0];
#pragma unroll
                        for (int it = 1; it < 8; it++) arg = (dl == it) ? sc[it] : arg;
                        arg = (dl == 8) ? m : arg;
                        const float em = expf(arg - mn);
                        const float f = row_lane<8>(em);
                        lsum *= f;
                        acc.x *= f;
                        acc.y *= f;
                        acc.z *= f;
                        acc.w *= f;
                        const float e[8] = {row_lane<0>(em), row_lane<1>(em), row_lane<2>(em), row_lane<3>(em),
                                            row_lane<4>(em), row_lane<5>(em), row_lane<6>(em), row_lane<7>(em)};
#pragma unroll
                        for (int it = 0; it < 8; it++) {
                            lsum += e[it];
                            acc.x += e[it] * v4[it].x;
                            acc.y += e[it] * v4[it].y;
                            acc.z += e[it] * v4[it].z;
                            acc.w += e[it] * v4[it].w;
                        }
                        m = mn;
                    };
                    fetch(t0);  // in flight while q is on its way
                    const float touched = spare && round == 0 ? touch(seq, h, t0 + 32, t1) : 0.0f;
                    {
                        const unsigned at = static_cast<unsigned>(seq * D + h * HS + dl * 4) * 8u;
                        const unsigned tag = sb + 1u;
                        unsigned spins = 0;
                        for (;;) {
                            v4i u[6];
#pragma unroll
                            for (int i = 0; i < 6; i++)
                                u[i] = coherent_load16(rs, (i < 2 || newest) ? static_cast<unsigned>((c_q + (i >> 1) * D * B) * 8) + at + (i & 1) * 16 : kPastEnd);
                            bool ok = true;
#pragma unroll
                            for (int i = 0; i < 6; i++)
                                ok = ok && ((i >= 2 && !newest) || (u[i].y == static_cast<int>(tag) && u[i].w == static_cast<int>(tag)));
                            q4 = make_float4(__int_as_float(u[0].x), __int_as_float(u[0].z), __int_as_float(u[1].x), __int_as_float(u[1].z));
                            kn = make_float4(__int_as_float(u[2].x), __int_as_float(u[2].z), __int_as_float(u[3].x), __int_as_float(u[3].z));
                            vn = make_float4(__int_as_float(u[4].x), __int_as_float(u[4].z), __int_as_float(u[5].x), __int_as_float(u[5].z));
                            if (__all(ok)) break;
                            if (hopeless(spins)) {
                                give_up(tag);
                                break;
                            }
                        }
                    }
                    asm volatile("" ::"v"(touched));
                    for (int tb = t0; tb < t1; tb += 32) {
                        if (tb > t0) fetch(tb);
                        work(tb);
                    }
                }
                lsum += __shfl_xor(lsum, 16, kWave);
                lsum += __shfl_xor(lsum, 32, kWave);
#pragma unroll
                for (int o = 16; o < 64; o <<= 1) {
                    acc.x += __shfl_xor(acc.x, o, kWave);
                    acc.y += __shfl_xor(acc.y, o, kWave);
                    acc.z += __shfl_xor(acc.z, o, kWave);
                    acc.w += __shfl_xor(acc.w, o, kWave);
                }
                float(*mine)[68] = part[(l * rounds + round) & 1][half];
                if (lane < 16) reinterpret_cast<float4*>(&mine[wv][4])[lane] = acc;
                if (lane == 0) {
                    mine[wv][0] = m;
                    mine[wv][1] = lsum;
                }
                __syncthreads();
                if (live && wv == 0) {
                    float M = -INFINITY, L = 0.0f, o = 0.0f;
                    for (int q = 0; q < 4; q++) M = fmaxf(M, mine[q][0]);
                    for (int q = 0; q < 4; q++) {
                        const float f = expf(mine[q][0] - M);
                        L += mine[q][1] * f;
                        o += mine[q][4 + lane] * f;
                    }
                    if (nchunk == 1) {
                        publish(seq, h, o * (1.0f / L));
                    } else if (ck > 0) {
                        Cell* out = p.cells + c_part + item * 66;
                        cell_put(out + 2 + lane, o, sb + 6u);
                        if (lane == 0) {
                            cell_put(out, M, sb + 6u);
                            cell_put(out + 1, L, sb + 6u);
                        }
                    } else if (ROUNDS) {
                        held[round][half][2 + lane] = o;
                        held[round][half][0] = M;
                        held[round][half][1] = L;
                    } else {
                        fold(item, M, L, o);
                    }
                }
                __syncthreads();  // nobody's loads go out in front of these stores
            }
            if (ROUNDS && nchunk > 1) {
                if (wv == 0) {
                    for (int round = 0; round < rounds; round++) {
                        const int item = order + (2 * round + half) * G;
                        if (item < items && item % nchunk == 0)
                            fold(item, held[round][half][0], held[round][half][1], held[round][half][2 + lane]);
                    }
                }
                __syncthreads();
            }
        }

        if (owner) {
            // ===== x += b_o + attn @ W_o
            const int n = wg * 16 + ej;
            float4 b[ND], a[ND];
            fetch_rows(w.wo, D, wg * 16, wave * (D / KW), b);
            float b0 = 0.0f, b1 = 0.0f, b20 = 0.0f, b21 = 0.0f;
            if (e_live) {
                b0 = w.bo[n];
                b1 = w.bo[n + 1];
                if (!MODERN) {
                    b20 = w.b2[n];
                    b21 = w.b2[n + 1];
                }
            }
            to_operands(b);
            poll_rows(c_at, wave * (D / KW), sb + 2u, a);
            v4f acc = {0.f, 0.f, 0.f, 0.f};
            multiply(a, b, acc);
            leave(1, 0, acc);
            __syncthreads();
            if (e_live) {
                float v0, v1;
                sum_pair(1, 0, v0, v1);
                r0 = (r0 + b0) + v0;
                r1 = (r1 + b1) + v1;
                cell_put2(rs, c_mid + operand_cell(n, ei, B), r0, r1, sb + 3u);
            }
            __syncthreads();
            // ===== x += (b2 +) hidden @ W2: the rows of W2 are on their way while the others form the
            // hidden values
            float4 b2[NF];
            fetch_rows(w.w2, F, wg * 16, wave * (F / KW), b2);
            to_operands(b2);
            acc = v4f{0.f, 0.f, 0.f, 0.f};
            constexpr int NR = RP == 16 ? 8 : NF;  // blocks per round of polls
            static_assert(NF % NR == 0, "whole rounds");
#pragma unroll
            for (int q = 0; q < NF / NR; q++) {
                float4 ah[NR], bh[NR];
                poll_rows(c_hid, wave * (F / KW) + q * NR * 16, sb + 4u, ah);
#pragma unroll
                for (int i = 0; i < NR; i++) bh[i] = b2[q * NR + i];
                multiply(ah, bh, acc);
            }
            leave(0, 0, acc);
            __syncthreads();
            if (e_live) {
                float v0, v1;
                sum_pair(0, 0, v0, v1);
                r0 = (r0 + b20) + v0;
                r1 = (r1 + b21) + v1;
                if (l + 1 < p.L) cell_put2(rs, c_x + operand_cell(n, ei, B), r0, r1, sb + 5u);
                else *reinterpret_cast<float2*>(p.x + static_cast<size_t>(ei) * D + n) = make_float2(r0, r1);
            }
            __syncthreads();
        } else if (u1 < T1) {
            // ===== norm2 + FFN1
            const bool two = u1 + NO < T1;
            float4 b[ND], bb[ND], a[ND], gain[ND], shift[ND];
            fetch_rows(w.w1, D, u1 * 16, wave * (D / KW), b);
            if (two) fetch_rows(w.w1, D, (u1 + NO) * 16, wave * (D / KW), bb);
            else {
#pragma unroll
                for (int i = 0; i < ND; i++) bb[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
            fetch_norm(w.g2, w.be2, gain, shift);
            float bias[4] = {0.f, 0.f, 0.f, 0.f};
            if (!MODERN && e_live) {
                bias[0] = w.b1[u1 * 16 + ej];
                bias[1] = w.b1[u1 * 16 + ej + 1];
                if (two) {
                    bias[2] = w.b1[(u1 + NO) * 16 + ej];
                    bias[3] = w.b1[(u1 + NO) * 16 + ej + 1];
                }
            }
            to_operands(b);
            if (two) to_operands(bb);
            poll_rows(c_mid, wave * (D / KW), sb + 3u, a);
            norm_rows(a, gain, shift, 1);
            v4f acc = {0.f, 0.f, 0.f, 0.f}, acc2 = {0.f, 0.f, 0.f, 0.f};
            multiply(a, b, acc);
            leave(1, 0, acc);
            if (two) {
                multiply(a, bb, acc2);
                leave(1, 1, acc2);
            }
            __syncthreads();
            if (e_live) {
                float r = 1.0f;
                if (MODERN) r = rms(1);
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    if (t == 1 && !two) break;
                    const int n = (u1 + t * NO) * 16 + ej;
                    float v0, v1;
                    sum_pair(1, t, v0, v1);
                    if (MODERN) {
                        v0 *= r;
                        v1 *= r;
                        cell_put(p.cells + c_hid + operand_cell(n >> 1, ei, B), v1 * silu(v0), sb + 4u);
                    } else {
                        cell_put2(rs, c_hid + operand_cell(n, ei, B), gelu_tanh(v0 + bias[2 * t]), gelu_tanh(v1 + bias[2 * t + 1]), sb + 4u);
                    }
                }
            }
            __syncthreads();
        }
        // (once per layer, and not in front of a phase's stores: behind an abandoned wait the layer goes on with
        // values that nobody will use)
        if (g_wait_abandoned) return;
    }
}

}  // namespace gh
