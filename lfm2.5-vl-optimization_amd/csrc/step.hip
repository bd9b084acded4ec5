// The non-matmul ops of one LFM2 decode step on gfx950, each as one or two launches over the runtime's static buffers:
//   attn_step   q / k head RMSNorm and rotary embedding, the new key and value into the cache, attention over it
//   conv_step   the gated short convolution: B x into its ring of the last inputs, the newest output, the gate C
//   embed_step  the residual stream's first value: the input tokens' embedding rows
//   step_tail   the end of the step: logits copy, greedy token of the unblocked logits, its output row, the counters
//
// Reference: the decode step's fused ops of src/lfm2opt/runtime.py:246-294 (its CUDA kernels of kernels/lfm2_decode.cu).
#include "common.hpp"
#include "status.hpp"

#include <algorithm>

namespace lfm2q {
namespace {

// ------------------------------------------------------------------------------------------------ attention
// One workgroup of 256 threads per (split, kv head, part of its query heads, batch row): G of the kv head's `grp` query
// heads against `chunks` consecutive chunks of PC cache positions, online softmax over the chunks, everything in fp32
// from the bf16 operands. The position is read on the device (ctr[0]), so one captured graph serves every position;
// chunks past it are not read. The workgroup of part 0 whose split holds the position writes the new key and value.
//
// What bounds it: latency, not bytes (200 positions of one kv head are 50 KiB), so every load of a chunk is issued
// before anything waits: thread t holds the keys of positions 8 (t % 32) .. + 7 for the eight dims 8 (t / 32) .. + 7
// (the cache keeps keys transposed, [hd, max_len]: 16 bytes are 8 positions of one dim, a wavefront load two whole
// 512-byte runs) and the values of 8 dims at positions t / 8 + 32 i, while the four wavefronts normalize and rotate the
// heads. The next chunk's loads go out as each register set is consumed. MI355X, 32 heads over 8, batch 1, in a graph:
// 4.9 us at 200 positions and 8.7 at 3,001, in place of the eleven PyTorch launches (norm, swap, products, two cache
// writes, scores, softmax, values) whose kernels took 32 and 43 us.
constexpr int HD = 64;   // head_dim
constexpr int PC = 256;  // cache positions per chunk

// The step's cache position, -1 outside the cache (its output is NaN then, and nothing else is read or written).
__device__ __forceinline__ int cache_pos(const int64_t *__restrict__ ctr, int max_len) {
    const int64_t p = ctr[0];
    return p < 0 || p >= max_len ? -1 : (int)p;
}

// head row `row` (q heads, then k heads) of the projection, normalized and rotated; lane d holds dim d. qkw: the head
// weights w [rows, 64], then [rows, 64] of (-w[32:], w[:32]), so rope(n w) = n (w cos) + swap(n) ((-w[32:], w[:32]) sin)
__device__ __forceinline__ float rope_head(float h, const float *__restrict__ qkw, int row, int rows,
                                           const float *__restrict__ rope, int lane, float eps) {
    const float w = qkw[row * HD + lane], wb = qkw[(rows + row) * HD + lane];
    const float c = rope[lane], s = rope[HD + lane];
    const float n = h * (1.f / sqrtf(wave_sum(h * h) * (1.f / HD) + eps));
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(n), __float_as_uint(n), false, false);
    // both halves of the swapped pair hold n of the other 32 lanes in one of the two results
    const float other = __uint_as_float(lane < 32 ? sw[1] : sw[0]);
    return n * (w * c) + other * (wb * s);
}

template <int G>
__global__ __launch_bounds__(256) void attn_step_kernel(const uint16_t *__restrict__ qkv, const float *__restrict__ qkw,
                                                        const float *__restrict__ rope, const int64_t *__restrict__ ctr,
                                                        uint16_t *kc, uint16_t *vc, uint16_t *__restrict__ out,
                                                        float *__restrict__ part, int nkv, int grp, int max_len,
                                                        int chunks, int splits, float scale_log2, float eps) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int split = blockIdx.x, kv = blockIdx.y % nkv, b = blockIdx.z;
    const int h0 = kv * grp + (blockIdx.y / nkv) * G;  // this workgroup's first query head
    const int nh = nkv * grp, ld = (nh + 2 * nkv) * HD;
    const int pos = cache_pos(ctr, max_len);
    if (pos < 0) {
        if (split == 0)
            for (int i = t; i < G * HD; i += 256) out[((size_t)b * nh + h0) * HD + i] = 0x7fff;
        return;
    }
    int p0 = split * chunks * PC;
    if (p0 > pos) return;  // uniform; the combine pass skips this split as well
    const int last = min(pos, p0 + chunks * PC - 1);  // this workgroup's last position
    const bool mine = last == pos;                    // it holds the new position
    kc += ((size_t)b * nkv + kv) * HD * max_len;
    vc += ((size_t)b * nkv + kv) * (size_t)max_len * HD;
    qkv += (size_t)b * ld;
    const uint16_t *vnew = qkv + (nh + nkv + kv) * HD;

    const int kp = 8 * (t & 31), kd = 8 * (t >> 5);  // keys: positions p0 + kp .. + 7, dims kd .. + 7
    const int vd = 8 * (t & 7), vr = t >> 3;         // values: dims vd .. + 7, positions p0 + vr + 32 i
    v4i kr[8], vv[8];
    auto load_k = [&](int p) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            kr[j] = p + kp <= last ? ld16(kc + (size_t)(kd + j) * max_len + p + kp) : v4i{0, 0, 0, 0};
    };
    auto load_v = [&](int p) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int q = p + vr + 32 * i;
            vv[i] = q <= last ? ld16((q == pos ? vnew : vc + (size_t)q * HD) + vd) : v4i{0, 0, 0, 0};
        }
    };
    load_k(p0);
    load_v(p0);

    __shared__ float qs[G][HD], kn[HD], snew[G], wm[4][G], wl[4][G];
    __shared__ float red[4 * G * PC > 32 * G * HD ? 4 * G * PC : 32 * G * HD];  // score partials, then value partials
    __shared__ float ps[PC][G];
    for (int h = wave; h < G + (mine ? 1 : 0); h += 4) {
        const int row = h < G ? h0 + h : nh + kv;
        const float x = rope_head(bf2f(qkv[row * HD + lane]), qkw, row, nh + nkv, rope + (size_t)pos * 2 * HD, lane, eps);
        if (h < G) {
            qs[h][lane] = x * scale_log2;
        } else {
            const uint32_t r = f2bf(x);
            kn[lane] = bf2f(r);
            if ((int)blockIdx.y < nkv) {
                kc[(size_t)lane * max_len + pos] = (uint16_t)r;
                vc[(size_t)pos * HD + lane] = vnew[lane];
            }
        }
    }
    __syncthreads();
    if (mine)
        for (int h = wave; h < G; h += 4) {
            const float s = wave_sum(qs[h][lane] * kn[lane]);
            if (lane == 0) snew[h] = s;
        }

    float m[G], l[G], acc[G][8];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        m[g] = -__builtin_inff();
        l[g] = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[g][e] = 0.f;
    }
    for (; p0 <= last; p0 += PC) {
        {
            float sc[G][8];
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int e = 0; e < 8; ++e) sc[g][e] = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const float qv = qs[g][kd + j];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        sc[g][2 * e] = __builtin_fmaf(qv, bf2f_lo((uint32_t)kr[j][e]), sc[g][2 * e]);
                        sc[g][2 * e + 1] = __builtin_fmaf(qv, bf2f_hi((uint32_t)kr[j][e]), sc[g][2 * e + 1]);
                    }
                }
            if (p0 + PC <= last) load_k(p0 + PC);
            // the wavefront's two 8-dim halves meet by a 32-lane swap: lanes 0-31 keep positions e < 4, 32-63 e >= 4
#pragma unroll
            for (int g = 0; g < G; ++g) {
                v4f r;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(sc[g][e]),
                                                                    __float_as_uint(sc[g][e + 4]), false, false);
                    r[e] = __uint_as_float(s[0]) + __uint_as_float(s[1]);
                }
                *reinterpret_cast<v4f *>(&red[(wave * G + g) * PC + kp + 4 * (lane >> 5)]) = r;
            }
        }
        __syncthreads();
        float s[G];
        const int p = p0 + t;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            s[g] = (red[g * PC + t] + red[(G + g) * PC + t]) + (red[(2 * G + g) * PC + t] + red[(3 * G + g) * PC + t]);
            if (p == pos) s[g] = snew[g];  // (a stale or half-written key is never used)
            if (p > last) s[g] = -__builtin_inff();
            const float w = wave_max(s[g]);
            if (lane == 0) wm[wave][g] = w;
        }
        __syncthreads();
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const float mn = fmaxf(m[g], fmaxf(fmaxf(wm[0][g], wm[1][g]), fmaxf(wm[2][g], wm[3][g])));
            const float a = __builtin_amdgcn_exp2f(m[g] - mn);  // 0 at the first chunk
            m[g] = mn;
            const float e = __builtin_amdgcn_exp2f(s[g] - mn);
            l[g] = l[g] * a + e;
            ps[t][g] = e;
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[g][i] *= a;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            float pg[G];
#pragma unroll
            for (int g = 0; g < G; ++g) pg[g] = ps[vr + 32 * i][g];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float lo = bf2f_lo((uint32_t)vv[i][e]), hi = bf2f_hi((uint32_t)vv[i][e]);
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    acc[g][2 * e] = __builtin_fmaf(pg[g], lo, acc[g][2 * e]);
                    acc[g][2 * e + 1] = __builtin_fmaf(pg[g], hi, acc[g][2 * e + 1]);
                }
            }
        }
        if (p0 + PC <= last) load_v(p0 + PC);
        // (the next chunk's writes to red, wm and ps each come after a barrier that follows these reads)
    }
    // the row sums and the 32 value partials of each head
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const float w = wave_sum(l[g]);
        if (lane == 0) wl[wave][g] = w;
#pragma unroll
        for (int h = 0; h < 2; ++h)
            *reinterpret_cast<v4f *>(&red[(vr * G + g) * HD + vd + 4 * h]) =
                v4f{acc[g][4 * h], acc[g][4 * h + 1], acc[g][4 * h + 2], acc[g][4 * h + 3]};
    }
    __syncthreads();
    for (int i = t; i < G * HD; i += 256) {
        const int g = i >> 6, d = i & 63;
        float o = 0.f;
#pragma unroll 8
        for (int r = 0; r < 32; ++r) o += red[(r * G + g) * HD + d];
        const float lt = (wl[0][g] + wl[1][g]) + (wl[2][g] + wl[3][g]);
        if (G > 1 || splits == 1) {
            out[((size_t)b * nh + h0 + g) * HD + d] = (uint16_t)f2bf(o / lt);
        } else {
            // partial (head, split): 64 unnormalized outputs, then its maximum and row sum (several splits: G = 1)
            float *pp = part + (((size_t)b * nh + h0) * splits + split) * (HD + 2);
            pp[d] = o;
            if (d == 0) pp[HD] = m[0], pp[HD + 1] = lt;
        }
    }
}

// The splits' partials of one head per wavefront, lane d holding dim d.
__global__ __launch_bounds__(256) void attn_combine_kernel(const float *__restrict__ part,
                                                           const int64_t *__restrict__ ctr, uint16_t *__restrict__ out,
                                                           int heads, int max_len, int chunks, int splits) {
    const int lane = threadIdx.x & 63;
    const int row = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));  // (batch row, head)
    if (row >= heads) return;
    const int pos = cache_pos(ctr, max_len);
    if (pos < 0) return;  // attn_step_kernel has written NaN
    const int n = pos / (chunks * PC) + 1;  // splits that hold positions
    const float *pp = part + (size_t)row * splits * (HD + 2);
    // lane i takes split i's maximum and sum (splits <= 64); the first 16 splits' outputs are in flight with them
    const float mi = pp[min(lane, n - 1) * (HD + 2) + HD], li = pp[min(lane, n - 1) * (HD + 2) + HD + 1];
    float o = 0.f, v[16];
    auto load = [&](int i0) {
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = pp[min(i0 + j, n - 1) * (HD + 2) + lane];
    };
    load(0);
    const float w = lane < n ? __builtin_amdgcn_exp2f(mi - wave_max(mi)) : 0.f;
    const float lt = wave_sum(w * li);
    for (int i = 0; i < n; i += 16) {
        float u[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) u[j] = v[j];
        if (i + 16 < n) load(i + 16);
#pragma unroll
        for (int j = 0; j < 16; ++j) o = __builtin_fmaf(lane_read(w, min(i + j, 63)), i + j < n ? u[j] : 0.f, o);
    }
    out[(size_t)row * HD + lane] = (uint16_t)f2bf(o / lt);
}

struct AttnShape {
    int chunks, splits, heads;  // chunks of PC positions and query heads per workgroup, splits of the positions
};
// First the query heads of a kv head over workgroups (each reads the kv head's cache again, from the L2) while that
// leaves no more workgroups than CUs: the arithmetic of four heads is half of a workgroup's time. Then the positions:
// about two workgroups a CU and at most 64 splits (the combine pass's lanes), but no split for two chunks or where
// fewer than four would come of it, which the combine pass (a launch, ~2.5 us) outweighs. Several heads a workgroup mean more
// than half as many workgroups as CUs, so at most three splits: they never come with several splits. MI355X, 32 heads over 8, us in
// a graph (rows, positions: heads per workgroup 1 / 2 / 4): 1, 200 4.9 / 5.6 / 7.0; 1, 400 6.5 / 7.6 / 10.0 (two splits
// 7.4 / 8.0 / 9.5); 1, 3001 in 16 splits 8.7 / 8.8 / 10.3 (8 splits 9.8, one 23.7); 16, 1000 13.5 / 13.3 / 17.7 (two
// splits 18.1 / 14.3 / 15.6); 64, 2000 90 / 63 / 58 (two splits 100 / 69 / 62).
inline AttnShape attn_shape(int B, int nkv, int grp, int max_len) {
    const int total = (max_len + PC - 1) / PC;
    int heads = grp;
    while (heads > 1 && (long)B * nkv * (grp / heads) * 2 <= device_cus()) heads /= 2;
    const int want = (int)std::min<long>(64, 2 * device_cus() / ((long)B * nkv * (grp / heads)));
    int splits = heads > 1 || total <= 2 || want < 4 ? 1 : std::min(total, want);
    const int chunks = (total + splits - 1) / splits;
    splits = (total + chunks - 1) / chunks;
    return {chunks, splits, heads};
}

// ------------------------------------------------------------------------------------------------ short convolution
// Thread: 4 channels of one batch row. ring [L, B, H] holds B x of the last L positions, position p in row p mod L; at
// position p ring row s holds p - (p - s) mod L, which tap L - 1 - (p - s) mod L multiplies (wt [L, H]). Rounded as
// transformers' bf16 step: B x, each tap's product, their fp32 sum (in ring order), with the bias, and times C. Latency:
// a few loads deep, so few channels per thread and many workgroups. The three-layer INT4 step lost 23 us with it, two
// layers of six PyTorch launches (~14 us of kernels each) against two of this one (~2 us).
constexpr int CONV_MAX = 8;  // longest ring

template <int L>
__global__ __launch_bounds__(64) void conv_step_kernel(const uint16_t *__restrict__ bcx, uint16_t *__restrict__ ring,
                                                       const uint16_t *__restrict__ wt,
                                                       const uint16_t *__restrict__ bias,
                                                       const int64_t *__restrict__ ctr, uint16_t *__restrict__ out,
                                                       int B, int H) {
#pragma clang fp contract(off)
    const int c = 4 * (blockIdx.x * 64 + threadIdx.x), b = blockIdx.y;
    if (c >= H) return;
    const uint16_t *row = bcx + (size_t)b * 3 * H + c;
    const uint2 vb = *reinterpret_cast<const uint2 *>(row), vc = *reinterpret_cast<const uint2 *>(row + H),
                vx = *reinterpret_cast<const uint2 *>(row + 2 * H);
    uint2 rv[L], wv[L];
#pragma unroll
    for (int s = 0; s < L; ++s) {
        rv[s] = *reinterpret_cast<const uint2 *>(ring + ((size_t)s * B + b) * H + c);
        wv[s] = *reinterpret_cast<const uint2 *>(wt + (size_t)s * H + c);
    }
    const uint2 bv = bias ? *reinterpret_cast<const uint2 *>(bias + c) : make_uint2(0, 0);
    const int r = (int)((ctr[0] % L + L) % L);
    const uint2 u = make_uint2(pack_bf16x2(bf2f_lo(vb.x) * bf2f_lo(vx.x), bf2f_hi(vb.x) * bf2f_hi(vx.x)),
                               pack_bf16x2(bf2f_lo(vb.y) * bf2f_lo(vx.y), bf2f_hi(vb.y) * bf2f_hi(vx.y)));
    *reinterpret_cast<uint2 *>(ring + ((size_t)r * B + b) * H + c) = u;
    float y[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < L; ++s) {
        const uint2 v = s == r ? u : rv[s];
        const int tap = s <= r ? L - 1 - (r - s) : s - r - 1;
        uint2 w = wv[0];
#pragma unroll
        for (int k = 1; k < L; ++k)
            if (k == tap) w = wv[k];
        y[0] += rbf(bf2f_lo(v.x) * bf2f_lo(w.x));
        y[1] += rbf(bf2f_hi(v.x) * bf2f_hi(w.x));
        y[2] += rbf(bf2f_lo(v.y) * bf2f_lo(w.y));
        y[3] += rbf(bf2f_hi(v.y) * bf2f_hi(w.y));
    }
    const float bf[4] = {bf2f_lo(bv.x), bf2f_hi(bv.x), bf2f_lo(bv.y), bf2f_hi(bv.y)};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        y[e] = rbf(y[e]);
        if (bias) y[e] = rbf(y[e] + bf[e]);
    }
    *reinterpret_cast<uint2 *>(out + (size_t)b * H + c) =
        make_uint2(pack_bf16x2(bf2f_lo(vc.x) * y[0], bf2f_hi(vc.x) * y[1]),
                   pack_bf16x2(bf2f_lo(vc.y) * y[2], bf2f_hi(vc.y) * y[3]));
}

// ------------------------------------------------------------------------------------------------ embedding and tail
// Thread: 8 values of one token's row. A token outside the vocabulary gives NaN (nothing is read for it). Latency: two
// dependent loads and a store. MI355X, 2,048 wide: batch 16 3.6 us against 10.3 for index_select (batch 1 2.4 for both).
__global__ __launch_bounds__(64) void embed_step_kernel(const uint16_t *__restrict__ table,
                                                        const int64_t *__restrict__ tok, uint16_t *__restrict__ h, int H,
                                                        int V) {
    const int c = 8 * (blockIdx.x * 64 + threadIdx.x), b = blockIdx.y;
    if (c >= H) return;
    const int64_t id = tok[b];
    const v4i nan = {0x7fff7fff, 0x7fff7fff, 0x7fff7fff, 0x7fff7fff};
    *reinterpret_cast<v4i *>(h + (size_t)b * H + c) = id >= 0 && id < V ? ld16(table + (size_t)id * H + c) : nan;
}

// A logit and its index as one key whose unsigned order is torch.argmax's: the larger value first, NaN above all, the
// lower index among equals (-0 equals +0).
__device__ __forceinline__ uint64_t argmax_key(float v, uint32_t i) {
    const uint32_t u = __float_as_uint(v + 0.f);
    const uint32_t o = v != v ? 0xffffffffu : u ^ ((u >> 31) ? 0xffffffffu : 0x80000000u);
    return (uint64_t)o << 32 | (uint32_t)~i;
}
__device__ __forceinline__ uint64_t max64(uint64_t a, uint64_t b) { return a > b ? a : b; }

// One workgroup per (chunk of TAIL_N logits, batch row): fp32 copies of its logits, and its largest key to part [B,
// chunks]; the last workgroup to arrive reduces every row's keys and writes the tokens and counters. The partial keys
// pass between XCDs as relaxed agent-scope accesses (coherent without a fence), each complete before its arrival.
// arrived returns to 0, so the workspace is zeroed once. Latency: one round of loads, an arrival and a second round;
// MI355X, 65,536 logits: 4.9 us at batch 1 and 11.4 at 16, in place of five PyTorch launches of 39 and 41 us (fp32 copy
// 4.5, mask 4.6, argmax 21.3 in too few workgroups, output row 4.6, counters 3.9).
constexpr int TAIL_N = 2048;

__global__ __launch_bounds__(256) void step_tail_kernel(const uint16_t *__restrict__ logits,
                                                        const uint8_t *__restrict__ block, float *__restrict__ copy,
                                                        int64_t *__restrict__ tok, int64_t *__restrict__ out,
                                                        int64_t *__restrict__ ctr, uint64_t *part, uint32_t *arrived,
                                                        int B, int V, int max_new, int set_pos) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, chunks = gridDim.x;
    const int b = blockIdx.y, c = blockIdx.x * TAIL_N + 8 * t;
    __shared__ uint64_t best[4];
    __shared__ uint32_t order;
    uint64_t key = 0;
    if (c < V) {
        const v4i v = ld16(logits + (size_t)b * V + c);
        const uint2 m = *reinterpret_cast<const uint2 *>(block + c);
        float f[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) f[2 * e] = bf2f_lo((uint32_t)v[e]), f[2 * e + 1] = bf2f_hi((uint32_t)v[e]);
        if (copy) {
            v4f *o = reinterpret_cast<v4f *>(copy + (size_t)b * V + c);
            o[0] = v4f{f[0], f[1], f[2], f[3]};
            o[1] = v4f{f[4], f[5], f[6], f[7]};
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const bool masked = ((e < 4 ? m.x : m.y) >> (8 * (e & 3)) & 0xffu) != 0;
            key = max64(key, argmax_key(masked ? -__builtin_inff() : f[e], (uint32_t)(c + e)));
        }
    }
    auto wave_key = [](uint64_t k, int width) {
        for (int d = width / 2; d; d >>= 1) k = max64(k, (uint64_t)__shfl_xor((unsigned long long)k, d, 64));
        return k;
    };
    key = wave_key(key, 64);
    if (lane == 0) best[wave] = key;
    __syncthreads();
    if (t == 0) {
        key = max64(max64(best[0], best[1]), max64(best[2], best[3]));
        __hip_atomic_store(part + (size_t)b * chunks + blockIdx.x, key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        order = __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (order != (uint32_t)(chunks * B) - 1) return;
    // two rows per wavefront and pass, four passes' loads in flight
    const int64_t row = set_pos >= 0 ? 0 : ctr[1];
    for (int r0 = 2 * wave + (lane >> 5); r0 < B; r0 += 32) {
        uint64_t k[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            k[i] = 0;
            if (r0 + 8 * i < B)
                for (int j = lane & 31; j < chunks; j += 32)
                    k[i] = max64(k[i], __hip_atomic_load(part + (size_t)(r0 + 8 * i) * chunks + j, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_AGENT));
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = r0 + 8 * i;
            const uint64_t w = wave_key(k[i], 32);
            if (r < B && (lane & 31) == 0) {
                const int64_t id = (int64_t)(uint32_t)~(uint32_t)w;
                tok[r] = id;
                if (row >= 0 && row < max_new) out[row * B + r] = id;
            }
        }
    }
    __syncthreads();  // every wavefront has read the output row
    if (t == 0) {
        ctr[0] = set_pos >= 0 ? set_pos : ctr[0] + 1;
        ctr[1] = row + 1;
        __hip_atomic_store(arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

}  // namespace
}  // namespace lfm2q

using namespace lfm2q;

extern "C" size_t lfm2q_attn_step_workspace_bytes(int B, int n_heads, int n_kv, int max_len) {
    if (B < 1 || n_heads < 1 || n_kv < 1 || max_len < 1) return 0;
    const AttnShape s = attn_shape(B, n_kv, std::max(1, n_heads / n_kv), max_len);
    return s.splits == 1 ? 0 : (size_t)B * n_heads * s.splits * (HD + 2) * 4;
}

extern "C" int lfm2q_attn_step(const lfm2q_bf16 *qkv, const float *qk_w, const float *rope, const int64_t *ctr,
                               lfm2q_bf16 *k, lfm2q_bf16 *v, lfm2q_bf16 *out, int B, int n_heads, int n_kv, int head_dim,
                               int max_len, float scale, float eps, void *ws, size_t ws_bytes, lfm2q_stream_t stream) {
    LFM2Q_REQUIRE(qkv && qk_w && rope && ctr && k && v && out, LFM2Q_ERR_ARG, "attn_step: null pointer");
    LFM2Q_REQUIRE(head_dim == HD, LFM2Q_ERR_SHAPE, "attn_step: head_dim must be %d (%d)", HD, head_dim);
    LFM2Q_REQUIRE(B >= 1 && B <= 65535 && n_kv >= 1 && n_heads >= 1 && n_heads <= 65535 && n_heads % n_kv == 0, LFM2Q_ERR_SHAPE,
                  "attn_step: bad B / heads (%d, %d, %d)", B, n_heads, n_kv);
    LFM2Q_REQUIRE(max_len >= 8 && max_len % 8 == 0, LFM2Q_ERR_SHAPE, "attn_step: max_len must be a multiple of 8 (%d)",
                  max_len);
    LFM2Q_REQUIRE(aligned16(qkv) && aligned16(k) && aligned16(v), LFM2Q_ERR_ALIGN,
                  "attn_step: qkv, k and v must be 16-byte aligned");
    const int grp = n_heads / n_kv;
    LFM2Q_REQUIRE(grp == 1 || grp == 2 || grp == 4 || grp == 8, LFM2Q_ERR_SHAPE,
                  "attn_step: query heads per kv head must be 1, 2, 4 or 8 (%d)", grp);
    const AttnShape s = attn_shape(B, n_kv, grp, max_len);
    LFM2Q_REQUIRE(s.splits == 1 || (ws && ws_bytes >= (size_t)B * n_heads * s.splits * (HD + 2) * 4), LFM2Q_ERR_ARG,
                  "attn_step: workspace smaller than lfm2q_attn_step_workspace_bytes()");
    const hipStream_t st = (hipStream_t)stream;
    const dim3 grid(s.splits, n_kv * (grp / s.heads), B);
    float *part = static_cast<float *>(ws);
    const float sl = scale * 1.44269504088896341f;
#define LFM2Q_ATTN(G_)                                                                                            \
    case G_:                                                                                                      \
        attn_step_kernel<G_><<<grid, 256, 0, st>>>(qkv, qk_w, rope, ctr, k, v, out, part, n_kv, grp, max_len,     \
                                                   s.chunks, s.splits, sl, eps);                                  \
        break;
    switch (s.heads) {
        LFM2Q_ATTN(1)
        LFM2Q_ATTN(2)
        LFM2Q_ATTN(4)
        LFM2Q_ATTN(8)
    }
#undef LFM2Q_ATTN
    if (s.splits > 1)
        attn_combine_kernel<<<(B * n_heads + 3) / 4, 256, 0, st>>>(part, ctr, out, B * n_heads, max_len, s.chunks,
                                                                   s.splits);
    return launch_status("attn_step");
}

extern "C" int lfm2q_conv_step(const lfm2q_bf16 *bcx, lfm2q_bf16 *ring, const lfm2q_bf16 *wt, const lfm2q_bf16 *bias,
                               const int64_t *ctr, lfm2q_bf16 *out, int B, int H, int L, lfm2q_stream_t stream) {
    LFM2Q_REQUIRE(bcx && ring && wt && ctr && out, LFM2Q_ERR_ARG, "conv_step: null pointer");
    LFM2Q_REQUIRE(B >= 1 && B <= 65535 && H >= 4 && H % 4 == 0, LFM2Q_ERR_SHAPE,
                  "conv_step: need 1 <= B <= 65535 and H %% 4 == 0 (B=%d H=%d)", B, H);
    LFM2Q_REQUIRE(((((uintptr_t)bcx | (uintptr_t)ring | (uintptr_t)wt) | ((uintptr_t)bias | (uintptr_t)out)) & 7) == 0,
                  LFM2Q_ERR_ALIGN, "conv_step: tensors must be 8-byte aligned");
    const dim3 grid((H / 4 + 63) / 64, B);
    const hipStream_t st = (hipStream_t)stream;
#define LFM2Q_CONV(L_) \
    case L_: conv_step_kernel<L_><<<grid, 64, 0, st>>>(bcx, ring, wt, bias, ctr, out, B, H); break;
    switch (L) {
        LFM2Q_CONV(1)
        LFM2Q_CONV(2)
        LFM2Q_CONV(3)
        LFM2Q_CONV(4)
        LFM2Q_CONV(5)
        LFM2Q_CONV(6)
        LFM2Q_CONV(7)
        LFM2Q_CONV(8)
    default: return set_error(LFM2Q_ERR_SHAPE, "conv_step: need 1 <= L <= %d (%d)", CONV_MAX, L);
    }
#undef LFM2Q_CONV
    return launch_status("conv_step");
}

extern "C" int lfm2q_embed_step(const lfm2q_bf16 *table, const int64_t *tok, lfm2q_bf16 *h, int B, int H, int V,
                                lfm2q_stream_t stream) {
    LFM2Q_REQUIRE(table && tok && h, LFM2Q_ERR_ARG, "embed_step: null pointer");
    LFM2Q_REQUIRE(B >= 1 && B <= 65535 && H >= 8 && H % 8 == 0 && V >= 1, LFM2Q_ERR_SHAPE,
                  "embed_step: need 1 <= B <= 65535 and H %% 8 == 0 (B=%d H=%d V=%d)", B, H, V);
    LFM2Q_REQUIRE(aligned16(table) && aligned16(h), LFM2Q_ERR_ALIGN, "embed_step: tensors must be 16-byte aligned");
    embed_step_kernel<<<dim3((H / 8 + 63) / 64, B), 64, 0, (hipStream_t)stream>>>(table, tok, h, H, V);
    return launch_status("embed_step");
}

extern "C" size_t lfm2q_step_tail_workspace_bytes(int B, int V) {
    if (B < 1 || V < 1) return 0;
    return 8 + (size_t)B * ((V + TAIL_N - 1) / TAIL_N) * 8;
}

extern "C" int lfm2q_step_tail(const lfm2q_bf16 *logits, const uint8_t *block, float *copy, int64_t *tok, int64_t *out,
                               int64_t *ctr, int B, int V, int max_new, int set_pos, void *ws, size_t ws_bytes,
                               lfm2q_stream_t stream) {
    LFM2Q_REQUIRE(logits && block && tok && out && ctr && ws, LFM2Q_ERR_ARG, "step_tail: null pointer");
    LFM2Q_REQUIRE(B >= 1 && B <= 65535 && V >= 8 && V % 8 == 0 && max_new >= 1, LFM2Q_ERR_SHAPE,
                  "step_tail: need 1 <= B <= 65535, V %% 8 == 0 and max_new >= 1 (B=%d V=%d max_new=%d)", B, V, max_new);
    const int chunks = (V + TAIL_N - 1) / TAIL_N;
    LFM2Q_REQUIRE((int64_t)chunks * B < (1ll << 31), LFM2Q_ERR_SHAPE, "step_tail: B V too large");
    LFM2Q_REQUIRE(aligned16(logits) && aligned16(copy) && ((uintptr_t)block & 7) == 0 && ((uintptr_t)ws & 7) == 0,
                  LFM2Q_ERR_ALIGN, "step_tail: logits and copy must be 16-byte, block and ws 8-byte aligned");
    LFM2Q_REQUIRE(ws_bytes >= lfm2q_step_tail_workspace_bytes(B, V), LFM2Q_ERR_ARG,
                  "step_tail: workspace smaller than lfm2q_step_tail_workspace_bytes()");
    uint32_t *arrived = static_cast<uint32_t *>(ws);
    uint64_t *part = reinterpret_cast<uint64_t *>(static_cast<char *>(ws) + 8);
    step_tail_kernel<<<dim3(chunks, B), 256, 0, (hipStream_t)stream>>>(logits, block, copy, tok, out, ctr, part, arrived,
                                                                       B, V, max_new, set_pos);
    return launch_status("step_tail");
}
