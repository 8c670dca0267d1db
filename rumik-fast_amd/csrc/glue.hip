// Decode-step glue for gfx950 (reference engine/fused.py): everything between the GEMVs.
//
// All kernels read `pos` (int64) from device memory, so one captured graph serves every sequence length, and
// write only their outputs (no allocation, no host sync). Activations are fp16 or bf16 (`dt`), math is fp32 and
// each stored value is rounded once, at the same points as the reference's fused step.
#include "common.h"

namespace {

constexpr int kLnThreads = 256;
constexpr int kLnMaxPerThread = 32;  // H <= 8192

// sum over the block (every thread gets the total); `red` holds one float per wave
RK_DEV float block_sum(float v, float* red) {
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    __syncthreads();  // red may still be read by a previous call
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float t = 0.f;
    for (int i = 0; i < nw; ++i) t += red[i];
    return t;
}

// Cohere LayerNorm of the block's register copy xv (element i = tid + k*blockDim), written to h:
// d = x - mean, h = d * rsqrt(mean(d^2) + eps) * w (reference engine/rumik_int4.py:38-43, engine/fused.py:23-26)
RK_DEV void layernorm_store(const float (&xv)[kLnMaxPerThread], const void* __restrict__ w, void* __restrict__ h,
                            int dt, int H, float eps, float* red) {
    const int per = (H + blockDim.x - 1) / blockDim.x;
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < kLnMaxPerThread; ++k)
        if (k < per && threadIdx.x + k * blockDim.x < H) s += xv[k];
    const float mean = block_sum(s, red) / (float)H;
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < kLnMaxPerThread; ++k)
        if (k < per && threadIdx.x + k * blockDim.x < H) {
            const float d = xv[k] - mean;
            ss += d * d;
        }
    const float rstd = 1.0f / sqrtf(block_sum(ss, red) / (float)H + eps);
#pragma unroll
    for (int k = 0; k < kLnMaxPerThread; ++k) {
        const int i = threadIdx.x + k * blockDim.x;
        if (k < per && i < H) store_act(h, dt, (size_t)i, (xv[k] - mean) * rstd * load_act(w, dt, (size_t)i));
    }
}

RK_DEV float round_act(float v, int dt) {
    if (dt == RK_F16) return (float)(_Float16)v;
    if (dt == RK_BF16) return bf16_bits_to_f32(f32_to_bf16_bits(v));
    return v;
}

// x = dt(emb_q[tok] * emb_s[tok]); h = LN(x) * w        (reference engine/fused.py:16-27)
__global__ __launch_bounds__(kLnThreads) void embed_ln_kernel(const int64_t* __restrict__ tok,
                                                              const int8_t* __restrict__ eq,
                                                              const uint16_t* __restrict__ es,
                                                              const void* __restrict__ w, void* __restrict__ x,
                                                              void* __restrict__ h, int dt, int H, float eps) {
    __shared__ float red[16];
    const int64_t t = tok[0];
    const float sc = f16_bits_to_f32(es[t]);
    const int8_t* row = eq + (size_t)t * H;
    float xv[kLnMaxPerThread];
#pragma unroll
    for (int k = 0; k < kLnMaxPerThread; ++k) {
        const int i = threadIdx.x + k * blockDim.x;
        xv[k] = 0.f;
        if (i < H) {
            xv[k] = round_act((float)row[i] * sc, dt);
            store_act(x, dt, (size_t)i, xv[k]);
        }
    }
    layernorm_store(xv, w, h, dt, H, eps, red);
}

// x = dt(x + a + b) (fp32 sum, one rounding); h = LN(x) * w    (reference engine/fused.py:30-41)
__global__ __launch_bounds__(kLnThreads) void add_ln_kernel(void* __restrict__ x, const void* __restrict__ a,
                                                            const void* __restrict__ b, const void* __restrict__ w,
                                                            void* __restrict__ h, int dt, int H, float eps) {
    __shared__ float red[16];
    float xv[kLnMaxPerThread];
#pragma unroll
    for (int k = 0; k < kLnMaxPerThread; ++k) {
        const int i = threadIdx.x + k * blockDim.x;
        xv[k] = 0.f;
        if (i < H) {
            float v = load_act(x, dt, (size_t)i) + load_act(a, dt, (size_t)i);
            if (b) v += load_act(b, dt, (size_t)i);
            xv[k] = round_act(v, dt);
            store_act(x, dt, (size_t)i, xv[k]);
        }
    }
    layernorm_store(xv, w, h, dt, H, eps, red);
}

// One launch for everything after the fused projection (reference engine/fused.py:44-84). Block b:
//   b < NH + NKV        RoPE one q or k head (interleaved pairs) -> q_out or the k cache slot pos
//   b < NH + 2 NKV      copy one v head into the v cache slot pos
//   otherwise           act = silu(gate) * up for 256 MLP channels
__global__ __launch_bounds__(64) void post_kernel(const void* __restrict__ y, const int64_t* __restrict__ posp,
                                                  const void* __restrict__ cos_t, const void* __restrict__ sin_t,
                                                  void* __restrict__ kc, void* __restrict__ vc, void* __restrict__ qo,
                                                  void* __restrict__ act, int dt, int NH, int NKV, int HD, int S,
                                                  int inter, int rope) {
    const int b = blockIdx.x, tid = threadIdx.x;
    const int64_t pos = posp[0];
    if (b < NH + 2 * NKV && (pos < 0 || pos >= S)) return;  // no cache slot for this position: write nothing
    if (b < NH + NKV) {
        for (int j = tid; j < HD / 2; j += 64) {
            const float xe = load_act(y, dt, (size_t)b * HD + 2 * j);
            const float xo = load_act(y, dt, (size_t)b * HD + 2 * j + 1);
            float oe = xe, oo = xo;
            if (rope) {
                const float c = load_act(cos_t, dt, (size_t)pos * HD + 2 * j);
                const float s = load_act(sin_t, dt, (size_t)pos * HD + 2 * j);
                oe = xe * c - xo * s;
                oo = xo * c + xe * s;
            }
            if (b < NH) {
                store_act(qo, dt, (size_t)b * HD + 2 * j, oe);
                store_act(qo, dt, (size_t)b * HD + 2 * j + 1, oo);
            } else {
                const size_t base = ((size_t)(b - NH) * S + pos) * HD;
                store_act(kc, dt, base + 2 * j, oe);
                store_act(kc, dt, base + 2 * j + 1, oo);
            }
        }
    } else if (b < NH + 2 * NKV) {
        const int vh = b - NH - NKV;
        const size_t src = (size_t)(NH + NKV) * HD + (size_t)vh * HD;
        const size_t dst = ((size_t)vh * S + pos) * HD;
        for (int d = tid; d < HD; d += 64) store_act(vc, dt, dst + d, load_act(y, dt, src + d));
    } else {
        const size_t off = (size_t)(NH + 2 * NKV) * HD;
        const int i0 = (b - NH - 2 * NKV) * 256;
        for (int i = i0 + tid; i < min(i0 + 256, inter); i += 64) {
            const float g = load_act(y, dt, off + i);
            const float u = load_act(y, dt, off + inter + i);
            store_act(act, dt, (size_t)i, g / (1.0f + __expf(-g)) * u);
        }
    }
}

// act[i] = silu(gate[i]) * up[i] (the MLP job of post on its own)
__global__ __launch_bounds__(256) void silu_mul_kernel(const void* __restrict__ gu, void* __restrict__ act, int dt,
                                                       int inter) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= inter) return;
    const float g = load_act(gu, dt, (size_t)i);
    const float u = load_act(gu, dt, (size_t)inter + i);
    store_act(act, dt, (size_t)i, g / (1.0f + __expf(-g)) * u);
}

// slots per split for n filled slots: ceil(n / nsplit) rounded up to a multiple of 8
RK_DEV int split_chunk(int n, int nsplit) { return ((n + nsplit - 1) / nsplit + 7) & ~7; }

// ---------------------------------------------------------------------------------------------- decode attention
// Both kernels are bound by latency, not bytes (2 MB of K / V per layer at 1001 slots): what counts is how many
// dependent loads and reductions stand in a row. Split + combine over 64 splits at 1001 slots, bf16, 16 / 4 heads, 12
// layers in one graph: 7.1 us per layer; with one slot per wave and round, and the combine reading its splits one
// after the other per dim, 28.8 us (8.6 + 19.8 us by kernel).
constexpr int kAttnWaves = 4;
constexpr int kAttnGroups = 4 * kAttnWaves;  // slots in flight per block: a 16-lane group each
constexpr int kAttnHeads = 4;                // heads merged through LDS at a time (32 KiB)

// 8 consecutive 16-bit values at element i of p: one 16-byte load (VEC: p 16-byte aligned, i % 8 == 0) or eight
// 2-byte ones
template <bool VEC>
RK_DEV u4_t load8(const void* __restrict__ p, size_t i) {
    const uint16_t* s = reinterpret_cast<const uint16_t*>(p) + i;
    if constexpr (VEC) {
        return *reinterpret_cast<const u4_t*>(s);
    } else {
        u4_t v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = (uint32_t)s[2 * e] | ((uint32_t)s[2 * e + 1] << 16);
        return v;
    }
}

template <bool BF16>
RK_DEV void widen8(u4_t d, float (&f)[8]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if constexpr (BF16) {
            f[2 * e] = __builtin_bit_cast(float, d[e] << 16);
            f[2 * e + 1] = __builtin_bit_cast(float, d[e] & 0xffff0000u);
        } else {
            f[2 * e] = (float)as_h2(d[e]).x;
            f[2 * e + 1] = (float)as_h2(d[e]).y;
        }
    }
}

// sum over the 16 lanes of a DPP row, in every lane
RK_DEV float row16_total(float v) {
    v += dpp<0x128>(v);
    v += dpp<0x124>(v);
    v += dpp<0x122>(v);
    v += dpp<0x121>(v);
    return v;
}

// Flash-decoding partials (reference engine/fused.py:120-169). Block (g, sp): KV head g, slots
// [sp*ch, min((sp+1)*ch, pos+1)), all REP query heads of g. A 16-lane group takes every 16th slot, lane j holding dims
// 8j .. 8j + 7 of q, k, v and of the running acc (HD = 128): one 16-byte load per slot and tensor, so a wave has four
// slots in one load and a split of up to 16 slots (any cache up to 1024 slots over 64 splits) needs one round trip
// to memory; the next round's K / V are loaded before a round is computed. Per slot: REP dot products (fp16:
// v_dot2_f32_f16, exact products; bf16: fp32 products of the widened values, so no bf16 value is narrowed to fp16
// range), four DPP steps each, an online-softmax update per head. The groups' partials are merged in LDS and written
// as (m, l, acc) per head and split; an empty split writes m = -inf, l = 0.
template <int REP, bool BF16, bool VEC>
__global__ __launch_bounds__(64 * kAttnWaves) void attn_split_kernel(const void* __restrict__ q,
                                                                      const void* __restrict__ kc,
                                                                      const void* __restrict__ vc,
                                                                      const int64_t* __restrict__ posp,
                                                                      float* __restrict__ po, float* __restrict__ pm,
                                                                      float* __restrict__ pl, int S, int nsplit,
                                                                      float scale) {
    constexpr int HD = 128, HB = REP < kAttnHeads ? REP : kAttnHeads;
    __shared__ float s_m[kAttnGroups][REP], s_l[kAttnGroups][REP];
    __shared__ __align__(16) float s_acc[kAttnGroups][HB][HD];
    const int g = blockIdx.x, sp = blockIdx.y, tid = threadIdx.x;
    const int sub = tid & 15, grp = tid >> 4;
    const int n = (int)max<int64_t>(min<int64_t>(posp[0] + 1, (int64_t)S), 0);
    const int ch = split_chunk(n, nsplit);
    const int start = sp * ch, end = min(start + ch, n);
    const size_t pi0 = (size_t)g * REP * nsplit + sp;  // head r's partial: pi0 + r * nsplit
    if (start >= end) {                                // block-uniform
        for (int i = tid; i < REP * HD; i += 64 * kAttnWaves) po[(pi0 + (size_t)(i / HD) * nsplit) * HD + i % HD] = 0.f;
        if (tid < REP) {
            pm[pi0 + (size_t)tid * nsplit] = -INFINITY;
            pl[pi0 + (size_t)tid * nsplit] = 0.f;
        }
        return;
    }
    const size_t kv = (size_t)g * S * HD + 8 * sub;
    auto slot = [&](int t) { return kv + (size_t)min(t, end - 1) * HD; };  // past the end: the last slot again, unused
    u4_t kr = load8<VEC>(kc, slot(start + grp)), vr = load8<VEC>(vc, slot(start + grp));

    u4_t qr[REP];
#pragma unroll
    for (int r = 0; r < REP; ++r) qr[r] = load8<VEC>(q, (size_t)(g * REP + r) * HD + 8 * sub);
    float m[REP], l[REP], acc[REP][8];
#pragma unroll
    for (int r = 0; r < REP; ++r) {
        m[r] = -INFINITY;
        l[r] = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[r][e] = 0.f;
    }
    for (int t0 = start; t0 < end; t0 += kAttnGroups) {
        const int t = t0 + grp;
        const u4_t kx = kr, vx = vr;
        if (t0 + kAttnGroups < end) {
            kr = load8<VEC>(kc, slot(t + kAttnGroups));
            vr = load8<VEC>(vc, slot(t + kAttnGroups));
        }
        float s[REP];
        if constexpr (BF16) {
            float kf[8];
            widen8<true>(kx, kf);
#pragma unroll
            for (int r = 0; r < REP; ++r) {
                float qf[8];
                widen8<true>(qr[r], qf);
                s[r] = qf[0] * kf[0];
#pragma unroll
                for (int e = 1; e < 8; ++e) s[r] = __builtin_fmaf(qf[e], kf[e], s[r]);
            }
        } else {
#pragma unroll
            for (int r = 0; r < REP; ++r) {
                s[r] = 0.f;
#pragma unroll
                for (int e = 0; e < 4; ++e) s[r] = dot2(as_h2(qr[r][e]), as_h2(kx[e]), s[r]);
            }
        }
        float vf[8];
        widen8<BF16>(vx, vf);
#pragma unroll
        for (int r = 0; r < REP; ++r) {
            const float sr = row16_total(s[r]) * scale;
            if (t < end) {
                const float mn = fmaxf(m[r], sr);
                const float ref = mn == -INFINITY ? 0.f : mn;  // a -inf score has weight 0
                const float alpha = __expf(m[r] - ref);        // m = -inf at the first slot: alpha = 0
                const float p = __expf(sr - ref);
                l[r] = l[r] * alpha + p;
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[r][e] = acc[r][e] * alpha + p * vf[e];
                m[r] = mn;
            }
        }
    }
#pragma unroll
    for (int r = 0; r < REP; ++r)
        if (sub == 0) {
            s_m[grp][r] = m[r];
            s_l[grp][r] = l[r];
        }
#pragma unroll
    for (int h0 = 0; h0 < REP; h0 += HB) {
        if (h0 > 0) __syncthreads();  // the previous heads' partials have been read
#pragma unroll
        for (int r = 0; r < HB; ++r) {
            f4_t* d = reinterpret_cast<f4_t*>(&s_acc[grp][r][8 * sub]);
            d[0] = f4_t{acc[h0 + r][0], acc[h0 + r][1], acc[h0 + r][2], acc[h0 + r][3]};
            d[1] = f4_t{acc[h0 + r][4], acc[h0 + r][5], acc[h0 + r][6], acc[h0 + r][7]};
        }
        __syncthreads();
        for (int i = tid; i < HB * HD; i += 64 * kAttnWaves) {
            const int r = i / HD, d = i % HD;
            float M = -INFINITY;
#pragma unroll
            for (int k = 0; k < kAttnGroups; ++k) M = fmaxf(M, s_m[k][h0 + r]);
            float L = 0.f, a = 0.f;
#pragma unroll
            for (int k = 0; k < kAttnGroups; ++k) {
                const float mk = s_m[k][h0 + r];
                const float wt = mk == -INFINITY ? 0.f : __expf(mk - M);
                L += wt * s_l[k][h0 + r];
                a += wt * s_acc[k][r][d];
            }
            const size_t pi = pi0 + (size_t)(h0 + r) * nsplit;
            po[pi * HD + d] = a;
            if (d == 0) {
                pm[pi] = M;
                pl[pi] = L;
            }
        }
    }
}

// out[h] = sum_i w_i acc_i / sum_i w_i l_i, w_i = exp(m_i - max m) over non-empty splits (fused.py:172-187).
// Block (head, 32 dims): thread = (split tid / 8 + 32 k, 4 dims 4 (tid % 8) ..): every wave reads all the head's m
// (a lane each) for their maximum while its own splits' acc are in flight, then the block's 32 partial sums per dim
// meet by lane swaps and LDS. VEC: po rows 16-byte aligned (HD % 4 == 0).
constexpr int kCombThreads = 256, kCombDims = 32;
template <bool VEC>
__global__ __launch_bounds__(kCombThreads) void attn_combine_kernel(const float* __restrict__ po,
                                                                    const float* __restrict__ pm,
                                                                    const float* __restrict__ pl,
                                                                    void* __restrict__ out, int dt, int HD,
                                                                    int nsplit) {
    __shared__ float s_num[kCombThreads / 64][kCombDims], s_den[kCombThreads / 64];
    const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int d0 = blockIdx.y * kCombDims + 4 * (tid & 7);
    const size_t base = (size_t)h * nsplit;
    auto load4 = [&](int i) {
        f4_t v = {0.f, 0.f, 0.f, 0.f};
        const float* p = po + (base + i) * HD + d0;
        if constexpr (VEC) {
            if (d0 < HD) v = *reinterpret_cast<const f4_t*>(p);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (d0 + e < HD) v[e] = p[e];
        }
        return v;
    };
    // the first 64 splits (all of them in the engines): loads first
    const int i0 = tid >> 3, i1 = i0 + 32, last = nsplit - 1;
    const f4_t a0 = load4(min(i0, last)), a1 = load4(min(i1, last));
    const float m0 = pm[base + min(i0, last)], m1 = pm[base + min(i1, last)];
    const float l0 = pl[base + min(i0, last)], l1 = pl[base + min(i1, last)];
    float M = -INFINITY;
    for (int i = lane; i < nsplit; i += 64) M = fmaxf(M, pm[base + i]);
    M = wave_max(M);
    f4_t num = {0.f, 0.f, 0.f, 0.f};
    float den = 0.f;
    auto add = [&](f4_t a, float m, float l) {
        const float wt = m == -INFINITY ? 0.f : __expf(m - M);
#pragma unroll
        for (int e = 0; e < 4; ++e) num[e] += wt * a[e];
        den += wt * l;
    };
    if (i0 < nsplit) add(a0, m0, l0);
    if (i1 < nsplit) add(a1, m1, l1);
    for (int i = i0 + 64; i < nsplit; i += 32) add(load4(i), pm[base + i], pl[base + i]);
    // over the wave's 8 splits (lane bits 3 .. 5), then the waves
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float v = num[e];
        num[e] = sum_xor<32>(sum_xor<16>(v + dpp<0x128>(v)));  // row_ror:8, then the lane swaps
    }
    den = sum_xor<32>(sum_xor<16>(den + dpp<0x128>(den)));
    if (lane < 8) {
#pragma unroll
        for (int e = 0; e < 4; ++e) s_num[wave][4 * lane + e] = num[e];
        if (lane == 0) s_den[wave] = den;
    }
    __syncthreads();
    const int d = blockIdx.y * kCombDims + tid;
    if (tid < kCombDims && d < HD) {
        float nu = 0.f, de = 0.f;
#pragma unroll
        for (int w = 0; w < kCombThreads / 64; ++w) {
            nu += s_num[w][tid];
            de += s_den[w];
        }
        store_act(out, dt, (size_t)h * HD + d, nu / de);
    }
}

__global__ void pos_advance_kernel(int64_t* pos) {
    if (threadIdx.x == 0) pos[0] += 1;
}

bool act_dt_ok(int dt) { return dt == RK_F16 || dt == RK_BF16; }

}  // namespace

extern "C" {

int rk_silu_mul(const void* gate_up, void* act, int act_dtype, int inter, rk_stream_t stream) {
    if (!gate_up || !act) return RK_ERR_NULL;
    if (inter <= 0) return RK_ERR_SHAPE;
    if (act_dtype != RK_F16 && act_dtype != RK_BF16 && act_dtype != RK_F32) return RK_ERR_DTYPE;
    hipLaunchKernelGGL(silu_mul_kernel, dim3((inter + 255) / 256), dim3(256), 0, (hipStream_t)stream, gate_up, act,
                       act_dtype, inter);
    return hipGetLastError() == hipSuccess ? RK_OK : RK_ERR_LAUNCH;
}

int rk_embed_ln(const int64_t* tok, const int8_t* emb_q, const uint16_t* emb_s, const void* ln_w, void* x, void* h,
                int act_dtype, int H, float eps, rk_stream_t stream) {
    if (!tok || !emb_q || !emb_s || !ln_w || !x || !h) return RK_ERR_NULL;
    if (H <= 0 || H > kLnThreads * kLnMaxPerThread) return RK_ERR_SHAPE;
    if (!act_dt_ok(act_dtype)) return RK_ERR_DTYPE;
    hipLaunchKernelGGL(embed_ln_kernel, dim3(1), dim3(kLnThreads), 0, (hipStream_t)stream, tok, emb_q, emb_s, ln_w, x,
                       h, act_dtype, H, eps);
    return hipGetLastError() == hipSuccess ? RK_OK : RK_ERR_LAUNCH;
}

int rk_add_ln(void* x, const void* a, const void* b, const void* ln_w, void* h, int act_dtype, int H, float eps,
              rk_stream_t stream) {
    if (!x || !a || !ln_w || !h) return RK_ERR_NULL;
    if (H <= 0 || H > kLnThreads * kLnMaxPerThread) return RK_ERR_SHAPE;
    if (!act_dt_ok(act_dtype)) return RK_ERR_DTYPE;
    hipLaunchKernelGGL(add_ln_kernel, dim3(1), dim3(kLnThreads), 0, (hipStream_t)stream, x, a, b, ln_w, h, act_dtype,
                       H, eps);
    return hipGetLastError() == hipSuccess ? RK_OK : RK_ERR_LAUNCH;
}

int rk_post(const void* y, const int64_t* pos, const void* cos_t, const void* sin_t, void* k_cache, void* v_cache,
            void* q_out, void* act, int act_dtype, int NH, int NKV, int HD, int S, int inter, int rope,
            rk_stream_t stream) {
    if (!y || !pos || !k_cache || !v_cache || !q_out || !act || (rope && (!cos_t || !sin_t))) return RK_ERR_NULL;
    if (NH <= 0 || NKV <= 0 || HD <= 0 || HD % 2 || S <= 0 || inter <= 0) return RK_ERR_SHAPE;
    if (!act_dt_ok(act_dtype)) return RK_ERR_DTYPE;
    const int blocks = NH + 2 * NKV + (inter + 255) / 256;
    hipLaunchKernelGGL(post_kernel, dim3(blocks), dim3(64), 0, (hipStream_t)stream, y, pos, cos_t, sin_t, k_cache,
                       v_cache, q_out, act, act_dtype, NH, NKV, HD, S, inter, rope);
    return hipGetLastError() == hipSuccess ? RK_OK : RK_ERR_LAUNCH;
}

int rk_attn_split(const void* q, const void* k_cache, const void* v_cache, const int64_t* pos, float* po, float* pm,
                  float* pl, int act_dtype, int NH, int NKV, int HD, int S, int nsplit, float scale,
                  rk_stream_t stream) {
    if (!q || !k_cache || !v_cache || !pos || !po || !pm || !pl) return RK_ERR_NULL;
    if (HD != 128 || NKV <= 0 || NH % NKV || S <= 0 || nsplit <= 0) return RK_ERR_SHAPE;
    if (!act_dt_ok(act_dtype)) return RK_ERR_DTYPE;
    const int rep = NH / NKV;
    const dim3 grid(NKV, nsplit);
    const hipStream_t s = (hipStream_t)stream;
    // rows of 256 bytes from 16-byte aligned bases take 16-byte loads; other pointers 2-byte ones
    const bool vec = !(((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15);
    const bool bf = act_dtype == RK_BF16;
#define RK_SPLIT(R, B, V)                                                                                             \
    hipLaunchKernelGGL((attn_split_kernel<R, B, V>), grid, dim3(64 * kAttnWaves), 0, s, q, k_cache, v_cache, pos, po, \
                       pm, pl, S, nsplit, scale)
#define RK_SPLIT_REP(R)                        \
    case R:                                    \
        if (bf && vec) RK_SPLIT(R, true, true);  \
        else if (bf) RK_SPLIT(R, true, false);   \
        else if (vec) RK_SPLIT(R, false, true);  \
        else RK_SPLIT(R, false, false);          \
        break;
    switch (rep) {
        RK_SPLIT_REP(1)
        RK_SPLIT_REP(2)
        RK_SPLIT_REP(4)
        RK_SPLIT_REP(8)
        default: return RK_ERR_SHAPE;
    }
#undef RK_SPLIT_REP
#undef RK_SPLIT
    return hipGetLastError() == hipSuccess ? RK_OK : RK_ERR_LAUNCH;
}

int rk_attn_combine(const float* po, const float* pm, const float* pl, const int64_t* pos, void* out, int act_dtype,
                    int NH, int HD, int nsplit, rk_stream_t stream) {
    if (!po || !pm || !pl || !out) return RK_ERR_NULL;
    if (NH <= 0 || HD <= 0 || nsplit <= 0) return RK_ERR_SHAPE;
    if (!act_dt_ok(act_dtype)) return RK_ERR_DTYPE;
    (void)pos;  // empty splits carry m = -inf and drop out of the merge, so the split lengths are not needed here
    const dim3 grid(NH, (HD + kCombDims - 1) / kCombDims);
    if (HD % 4 == 0 && !((uintptr_t)po & 15))
        hipLaunchKernelGGL(attn_combine_kernel<true>, grid, dim3(kCombThreads), 0, (hipStream_t)stream, po, pm, pl,
                           out, act_dtype, HD, nsplit);
    else
        hipLaunchKernelGGL(attn_combine_kernel<false>, grid, dim3(kCombThreads), 0, (hipStream_t)stream, po, pm, pl,
                           out, act_dtype, HD, nsplit);
    return hipGetLastError() == hipSuccess ? RK_OK : RK_ERR_LAUNCH;
}

int rk_pos_advance(int64_t* pos, rk_stream_t stream) {
    if (!pos) return RK_ERR_NULL;
    hipLaunchKernelGGL(pos_advance_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, pos);
    return hipGetLastError() == hipSuccess ? RK_OK : RK_ERR_LAUNCH;
}

}  // extern "C"
