// The transformer layer around the quantized projections, device-resident: RMSNorm (plain and
// fused with the residual add), RoPE with the KV-cache write, grouped-query attention over the
// cache, SwiGLU, the residual add, the KV-cache pool and the layer pipeline that chains them
// with the fused projection launches.
//
// Reference: src/kernels/rmsnorm.hip, rope.hip, attention.hip (gqa_online_softmax_kernel :35-123,
// DeviceKVCachePool :164-222, launch_forward_layer_cached_fp16 :603-695), mlp.hip.  Storage is
// fp16 and arithmetic fp32 with one rounding per stored value, as there.
//
// MI355X design:
//   * RMSNorm: one workgroup (4 waves) per row, 16-byte loads, wave64 DPP reductions.
//   * RoPE: one launch rotates q into its buffer, rotates k straight into the layer's K cache
//     at the token positions and copies v into the V cache (the reference copies K/V into the
//     pool separately); inverse frequencies come from the host in fp32, as in the reference.
//   * Attention of head_dim 64 and 128 runs on the matrix cores: 16-row tiles for decode and short
//     calls, 128-row tiles from 16 positions on, the keys split over workgroups where the row tiles
//     leave the chip idle.  Other head sizes: a wave owns (query row, query head, chunk of 64 keys) on
//     the vector ALUs.  Ranges are merged in a fixed order by a second pass (deterministic), skipped
//     for one range.
//   * SwiGLU and the residual add: 8 values per thread.
//   * Layer: q/k/v and gate/up each run as one fused projection launch (qmm_gemm_batch), all
//     kernels on the caller's stream with no host synchronisation; activations live in a
//     grow-only per-(device, stream) workspace.
#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "qmm_device.h"

namespace qmm {
namespace {

constexpr int kNormThreads = 256;
constexpr int kAttnChunk = 64;       // keys per attention chunk (one wave each)
constexpr int kMaxHeadDim = 256;
constexpr int kMaxRopePairs = kMaxHeadDim / 2;

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// fp32 acc + the dot product of two f16 pairs (v_dot2_f32_f16)
__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float acc) {
    h2v x, y;
    __builtin_memcpy(&x, &a, 4);
    __builtin_memcpy(&y, &b, 4);
    return __builtin_amdgcn_fdot2(x, y, acc, false);
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__device__ __forceinline__ float norm_weight(const void* w, int w_f32, int k) {
    // an F32 norm weight is rounded to f16 first, as the reference's host does
    if (w_f32) return static_cast<float>(static_cast<_Float16>(static_cast<const float*>(w)[k]));
    return static_cast<float>(static_cast<const _Float16*>(w)[k]);
}

// out[m] = half(v * rsqrt(mean(v^2) + eps) * w) with v = x[m] (res == nullptr) or
// v = half(x[m] + res[m]) (stored to h_out in the first pass and read back in the second, so
// h_out may alias x or res; out may alias x).  Each thread reads and writes only its own
// elements across the two passes.  Rows that do not fit rmsnorm_reg_kernel's registers.
__global__ __launch_bounds__(kNormThreads) void rmsnorm_kernel(const _Float16* x, const _Float16* res,
                                                              const void* __restrict__ w, int w_f32, _Float16* h_out,
                                                              _Float16* out, int K, float eps) {
    const int m = blockIdx.x;
    const size_t base = static_cast<size_t>(m) * K;
    const int tid = threadIdx.x;
    const bool vec = (K % 8) == 0;
    auto value = [&](int k) -> float {
        if (res == nullptr) return static_cast<float>(x[base + k]);
        return static_cast<float>(static_cast<_Float16>(static_cast<float>(x[base + k]) + static_cast<float>(res[base + k])));
    };
    float ss = 0.0f;
    if (vec) {
        for (int c = tid; c < K / 8; c += kNormThreads) {
            const h8 a = *reinterpret_cast<const h8*>(x + base + 8 * c);
            h8 v = a;
            if (res != nullptr) {
                const h8 r = *reinterpret_cast<const h8*>(res + base + 8 * c);
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = static_cast<_Float16>(static_cast<float>(a[e]) + static_cast<float>(r[e]));
                *reinterpret_cast<h8*>(h_out + base + 8 * c) = v;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float f = static_cast<float>(v[e]);
                ss += f * f;
            }
        }
    } else {
        for (int k = tid; k < K; k += kNormThreads) {
            const float f = value(k);
            if (res != nullptr) h_out[base + k] = static_cast<_Float16>(f);
            ss += f * f;
        }
    }
    __shared__ float part[kNormThreads / 64];
    ss = wave_sum(ss);
    if ((tid & 63) == 0) part[tid >> 6] = ss;
    __syncthreads();
    float tot = 0.0f;
#pragma unroll
    for (int i = 0; i < kNormThreads / 64; ++i) tot += part[i];
    const float scale = rsqrtf(tot / static_cast<float>(K) + eps);
    const _Float16* src = res == nullptr ? x : h_out;
    if (vec) {
        for (int c = tid; c < K / 8; c += kNormThreads) {
            const h8 v = *reinterpret_cast<const h8*>(src + base + 8 * c);
            h8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = static_cast<_Float16>(static_cast<float>(v[e]) * scale * norm_weight(w, w_f32, 8 * c + e));
            *reinterpret_cast<h8*>(out + base + 8 * c) = o;
        }
    } else {
        for (int k = tid; k < K; k += kNormThreads)
            out[base + k] = static_cast<_Float16>(static_cast<float>(src[base + k]) * scale * norm_weight(w, w_f32, k));
    }
}

// The same for K % 8 == 0 and K <= 2048 V: a thread holds its V vectors between the passes, so every load of
// the row (x, res, w) is requested at once and nothing is read twice; same sums in the same order.  w is
// read as vectors at any alignment.  Bound by its row traffic: 1023 rows of 8192, without and with a
// residual (33 and 67 MB), 9 and 13 us against 22 and 26 us with values read back and weights read one by one.
template <int V>
__global__ __launch_bounds__(kNormThreads) void rmsnorm_reg_kernel(const _Float16* x, const _Float16* res,
                                                                  const void* __restrict__ w, int w_f32, _Float16* h_out,
                                                                  _Float16* out, int K, float eps) {
    const size_t base = static_cast<size_t>(blockIdx.x) * K;
    const int tid = threadIdx.x;
    h8 v[V], r[V];
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const int c = min(tid + kNormThreads * i, K / 8 - 1);
        v[i] = *reinterpret_cast<const h8*>(x + base + 8 * c);
    }
    if (res != nullptr) {
#pragma unroll
        for (int i = 0; i < V; ++i) r[i] = *reinterpret_cast<const h8*>(res + base + 8 * min(tid + kNormThreads * i, K / 8 - 1));
#pragma unroll
        for (int i = 0; i < V; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) v[i][e] = static_cast<_Float16>(static_cast<float>(v[i][e]) + static_cast<float>(r[i][e]));
    }
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const int c = tid + kNormThreads * i;
        if (c < K / 8) {
            if (res != nullptr) *reinterpret_cast<h8*>(h_out + base + 8 * c) = v[i];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float f = static_cast<float>(v[i][e]);
                ss += f * f;
            }
        }
    }
    __shared__ float part[kNormThreads / 64];
    ss = wave_sum(ss);
    if ((tid & 63) == 0) part[tid >> 6] = ss;
    __syncthreads();
    float tot = 0.0f;
#pragma unroll
    for (int i = 0; i < kNormThreads / 64; ++i) tot += part[i];
    const float scale = rsqrtf(tot / static_cast<float>(K) + eps);
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const int c = tid + kNormThreads * i;
        if (c >= K / 8) continue;
        h8 wv;  // an F32 norm weight is rounded to f16 first, as the reference's host does
        if (w_f32) {
            float f[8];
            __builtin_memcpy(f, static_cast<const float*>(w) + 8 * c, 32);
#pragma unroll
            for (int e = 0; e < 8; ++e) wv[e] = static_cast<_Float16>(f[e]);
        } else {
            __builtin_memcpy(&wv, static_cast<const _Float16*>(w) + 8 * c, 16);
        }
        h8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = static_cast<_Float16>(static_cast<float>(v[i][e]) * scale * static_cast<float>(wv[e]));
        *reinterpret_cast<h8*>(out + base + 8 * c) = o;
    }
}

// out = half(x + r), 8 values per thread (n % 8 == 0) or one.
__global__ __launch_bounds__(256) void residual_add_kernel(const _Float16* __restrict__ x, const _Float16* __restrict__ r,
                                                          _Float16* __restrict__ out, int64_t n) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if ((n & 7) == 0) {
        if (8 * i >= n) return;
        const h8 a = *reinterpret_cast<const h8*>(x + 8 * i);
        const h8 b = *reinterpret_cast<const h8*>(r + 8 * i);
        h8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = static_cast<_Float16>(static_cast<float>(a[e]) + static_cast<float>(b[e]));
        *reinterpret_cast<h8*>(out + 8 * i) = o;
    } else if (i < n) {
        out[i] = static_cast<_Float16>(static_cast<float>(x[i]) + static_cast<float>(r[i]));
    }
}

// out = half(silu(g) * u), silu(g) = g / (1 + exp(-g)).
// y[r, i] = f16(f32(y[r, i]) + f32(b[i])) over `rows` rows of n values: a projection's bias added in
// fp32 to its fp16 output and rounded once (reference src/layer.py:274-282, 344-346).
__global__ __launch_bounds__(256) void bias_add_kernel(_Float16* __restrict__ y, const _Float16* __restrict__ b, int n,
                                                       int64_t total) {
    const int64_t stride = static_cast<int64_t>(gridDim.x) * 256;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < total; i += stride)
        y[i] = static_cast<_Float16>(static_cast<float>(y[i]) + static_cast<float>(b[i % n]));
}

__global__ __launch_bounds__(256) void swiglu_kernel(const _Float16* __restrict__ g, const _Float16* __restrict__ u,
                                                    _Float16* __restrict__ out, int64_t n) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    auto f = [](float gv, float uv) { return static_cast<_Float16>(gv / (1.0f + expf(-gv)) * uv); };
    if ((n & 7) == 0) {
        if (8 * i >= n) return;
        const h8 a = *reinterpret_cast<const h8*>(g + 8 * i);
        const h8 b = *reinterpret_cast<const h8*>(u + 8 * i);
        h8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = f(static_cast<float>(a[e]), static_cast<float>(b[e]));
        *reinterpret_cast<h8*>(out + 8 * i) = o;
    } else if (i < n) {
        out[i] = f(static_cast<float>(g[i]), static_cast<float>(u[i]));
    }
}

struct RopeFreq {
    float inv[kMaxRopePairs];
};

// Rotates pairs of q (n_q heads) into q_out and of k (n_k heads) into k_out, and copies v
// (n_k heads) into v_out; rows are token positions pos_offset + s.  q_out / k_out / v_out row
// strides are given in elements (the KV cache rows hold n_k heads).  A thread takes one pair of one
// position and every hg-th head of its block's range, so that an angle's sine and cosine serve all of
// them (1023 positions of 64 + 8 heads of 128: 15.0 us against 20.8 us with one thread per rotated pair).
// Block (x, y): ppb positions from x ppb, more than one where the heads leave threads idle (20000 positions of
// one head of 128: 7.3 us against 10.6 us with one), heads [y hpb, y hpb + hpb).
__global__ __launch_bounds__(256) void rope_kernel(const _Float16* q, _Float16* q_out, int n_q, const _Float16* k, _Float16* k_out,
                                                  const _Float16* v, _Float16* v_out, int n_k, int seq_len, int head_dim, int pos_offset,
                                                  int neox, int hpb, int hg, int ppb, RopeFreq fr) {
    const int half_dim = head_dim / 2;
    const int p = threadIdx.x % half_dim, gi = threadIdx.x / half_dim;
    const int s = blockIdx.x * ppb + gi / hg;
    if (gi >= hg * ppb || s >= seq_len) return;
    const float ang = static_cast<float>(pos_offset + s) * fr.inv[p];
    const float c = cosf(ang), sn = sinf(ang);
    const int i0 = neox ? p : 2 * p;
    const int i1 = neox ? p + half_dim : 2 * p + 1;
    const int end = min(n_q + n_k, static_cast<int>(blockIdx.y + 1) * hpb);
    for (int hh = blockIdx.y * hpb + gi % hg; hh < end; hh += hg) {
        const _Float16* src;
        _Float16* dst;
        if (hh < n_q) {
            src = q + (static_cast<size_t>(s) * n_q + hh) * head_dim;
            dst = q_out + (static_cast<size_t>(s) * n_q + hh) * head_dim;
        } else {
            const size_t at = (static_cast<size_t>(s) * n_k + (hh - n_q)) * head_dim;
            src = k + at;
            dst = k_out + at;
            if (v != nullptr) {
                v_out[at + i0] = v[at + i0];
                v_out[at + i1] = v[at + i1];
            }
        }
        const float a = static_cast<float>(src[i0]), b = static_cast<float>(src[i1]);
        dst[i0] = static_cast<_Float16>(a * c - b * sn);
        dst[i1] = static_cast<_Float16>(a * sn + b * c);
    }
}

// Attention, one wave per (query row m, query head h, key chunk c).  Lane l holds the D
// consecutive dimensions D*l .. D*l + D - 1 of the head (head_dim <= 64 D), so a key row is one
// coalesced read across the wave.  Keys are taken 8 at a time: the 8 K and V rows are loaded
// together (8 reads in flight per wave instead of one), the 8 dot products are reduced across
// the wave together, then the fp32 online softmax takes them in key order.  Partial results
// (running max, sum and unnormalised output), or the fp16 output when there is one chunk.
template <int D>
__global__ __launch_bounds__(256) void attention_kernel(const _Float16* __restrict__ Q, const _Float16* __restrict__ Kc,
                                                       const _Float16* __restrict__ Vc, _Float16* __restrict__ out,
                                                       float* __restrict__ part, int q_len, int kv_len, int heads,
                                                       int kv_heads, int head_dim, int start_pos, float scale, int causal,
                                                       int chunks) {
    constexpr int G = 8;  // keys per batch
    const int lane = threadIdx.x & 63;
    // wave-uniform (scalar registers), so the head, chunk and row arithmetic below is scalar
    const int64_t wave = static_cast<int64_t>(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t total = static_cast<int64_t>(q_len) * heads * chunks;
    if (wave >= total) return;
    // waves of one workgroup: consecutive heads of the same (m, c), so the query heads that share
    // a KV head (consecutive h) read the same keys
    const int h = static_cast<int>(wave % heads);
    const int64_t t = wave / heads;
    const int c = static_cast<int>(t % chunks);
    const int m = static_cast<int>(t / chunks);
    const int group = heads / kv_heads;
    const int kvh = h / group;
    const int n_keys = causal ? min(kv_len, start_pos + m + 1) : kv_len;
    const int s0 = c * kAttnChunk;
    const int s1 = min(n_keys, s0 + kAttnChunk);
    const bool full = head_dim == 64 * D;  // every lane owns D valid dims: vector reads
    const int d0 = D * lane;

    auto load = [&](const _Float16* p, float (&o)[D]) {
        if (full) {
            _Float16 v[D];
            __builtin_memcpy(v, p + d0, sizeof(v));
#pragma unroll
            for (int i = 0; i < D; ++i) o[i] = static_cast<float>(v[i]);
        } else {
#pragma unroll
            for (int i = 0; i < D; ++i) o[i] = d0 + i < head_dim ? static_cast<float>(p[d0 + i]) : 0.0f;
        }
    };
    float qv[D], acc[D];
    load(Q + (static_cast<size_t>(m) * heads + h) * head_dim, qv);
#pragma unroll
    for (int i = 0; i < D; ++i) acc[i] = 0.0f;
    float mx = -INFINITY, sum = 0.0f;
    const size_t row = static_cast<size_t>(kv_heads) * head_dim;
    const _Float16* kbase = Kc + static_cast<size_t>(kvh) * head_dim;
    const _Float16* vbase = Vc + static_cast<size_t>(kvh) * head_dim;
    for (int s = s0; s < s1; s += G) {
        const int n = min(G, s1 - s);
        float kk[G][D], vv[G][D];
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const size_t r = static_cast<size_t>(s + min(j, n - 1));  // rows past the end re-read the last
            load(kbase + r * row, kk[j]);
            load(vbase + r * row, vv[j]);
        }
        float dot[G];
#pragma unroll
        for (int j = 0; j < G; ++j) {
            dot[j] = 0.0f;
#pragma unroll
            for (int i = 0; i < D; ++i) dot[j] += qv[i] * kk[j][i];
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
#pragma unroll
            for (int j = 0; j < G; ++j) dot[j] += __shfl_xor(dot[j], o, 64);
#pragma unroll
        for (int j = 0; j < G; ++j) {
            if (j < n) {
                const float sc = dot[j] * scale;
                const float mn = fmaxf(mx, sc);
                const float a = expf(mx - mn);  // exp(-inf) = 0 for the first key
                const float e = expf(sc - mn);
                sum = sum * a + e;
#pragma unroll
                for (int i = 0; i < D; ++i) acc[i] = acc[i] * a + e * vv[j][i];
                mx = mn;
            }
        }
    }
    auto store = [&](auto* dst, auto cvt) {
        if (full) {
#pragma unroll
            for (int i = 0; i < D; ++i) dst[d0 + i] = cvt(acc[i]);
        } else {
#pragma unroll
            for (int i = 0; i < D; ++i)
                if (d0 + i < head_dim) dst[d0 + i] = cvt(acc[i]);
        }
    };
    if (chunks == 1) {
        const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
        store(out + (static_cast<size_t>(m) * heads + h) * head_dim, [&](float v) { return static_cast<_Float16>(v * inv); });
        return;
    }
    float* pp = part + static_cast<size_t>(wave) * (head_dim + 2);
    if (lane == 0) {
        pp[0] = mx;
        pp[1] = sum;
    }
    store(pp + 2, [](float v) { return v; });
}

// Attention for head_dim a multiple of 8 up to 128, one wave per (query row m, query head h, chunk
// of 64 keys), with lanes over keys for the scores and over dimensions for the output:
//   * lane j reads the whole K row of key s0 + j (16-byte loads, all in flight at once) and
//     forms q . k with v_dot2 on f16 pairs (q is the same for every lane);
//   * one wave max and one wave sum give the chunk's softmax statistics;
//   * lane l then owns dims 2l, 2l + 1 of the output, reads the V rows of all the chunk's keys at
//     once and accumulates p_j v_j with p_j broadcast from lane j.
// Output: partial results (max, sum, unnormalised output) as attention_kernel, or fp16 output
// when there is one chunk.
// With kRope (one query row, the decode step): Q, k_new and v_new are the projections before
// RoPE; each wave rotates its query into LDS, the new key (position start_pos) is rotated into LDS
// and stands in for its cache row, and the first query head of each KV head's group writes the
// rotated key and the value into the cache row.  No wave of the launch uses that row's cache
// contents: the new key's lane takes the rotated key from LDS and its value from v_new (a load
// of the row issued for a masked or replaced lane is discarded).
struct DecodeRope {
    const _Float16* k_new;  // [kv_heads][head_dim]
    const _Float16* v_new;
    _Float16* kc;           // the layer's K / V cache (rows of kv_heads * head_dim)
    _Float16* vc;
    int neox;
    float cs[kMaxRopePairs / 2], sn[kMaxRopePairs / 2];  // cos / sin of pair p's angle at the new position
};

template <bool kRope>
__global__ __launch_bounds__(256) void attention_keys_kernel(const _Float16* __restrict__ Q, const _Float16* __restrict__ Kc,
                                                            const _Float16* __restrict__ Vc, _Float16* __restrict__ out,
                                                            float* __restrict__ part, int q_len, int kv_len, int heads,
                                                            int kv_heads, int head_dim, int start_pos, float scale,
                                                            int causal, int chunks, DecodeRope dr) {
    constexpr int kMaxPairs = 64;  // head_dim <= 128
    const int lane = threadIdx.x & 63;
    // wave-uniform (scalar registers), so the head, chunk and row arithmetic below is scalar
    const int wl = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t wave = static_cast<int64_t>(blockIdx.x) * 4 + wl;
    const int64_t total = static_cast<int64_t>(q_len) * heads * chunks;
    if (wave >= total) return;
    const int h = static_cast<int>(wave % heads);
    const int64_t t = wave / heads;
    const int c = static_cast<int>(t % chunks);
    const int m = static_cast<int>(t / chunks);
    const int kvh = h / (heads / kv_heads);
    const int n_keys = causal ? min(kv_len, start_pos + m + 1) : kv_len;
    const int s0 = c * kAttnChunk;
    const int n = max(0, min(n_keys, s0 + kAttnChunk) - s0);  // keys of this chunk
    const int pairs = head_dim / 2;
    const size_t row = static_cast<size_t>(kv_heads) * head_dim;

    // scores: lane j <-> key s0 + j (lanes past the chunk re-read its first key and are masked)
    const uint32_t* qp = reinterpret_cast<const uint32_t*>(Q + (static_cast<size_t>(m) * heads + h) * head_dim);
    const int pos = start_pos + m;                       // the new key (kRope: m == 0)
    const int j_new = kRope && pos >= s0 && pos < s0 + kAttnChunk ? pos - s0 : -1;
    // The chunk's K and V rows are requested first: they do not depend on the rotation below, so
    // one memory round trip covers them, the query and the new key.
    // A dummy lane (and the new key's lane, which takes its key from LDS) reads a row below the
    // new key: s0 when the new key is not the chunk's first, else row 0 (pos > 0), else it is masked
    const int dummy = j_new == 0 ? 0 : s0;
    const int sj = lane < n && lane != j_new ? s0 + lane : (kRope ? min(dummy, max(pos - 1, 0)) : s0);
    const u32x4* kr = reinterpret_cast<const u32x4*>(Kc + static_cast<size_t>(sj) * row + static_cast<size_t>(kvh) * head_dim);
    u32x4 kv[kMaxPairs / 4];
#pragma unroll
    for (int i = 0; i < kMaxPairs / 4; ++i)
        if (4 * i < pairs) kv[i] = kr[i];
    // the chunk's V rows are requested together with the K rows (they do not depend on the scores):
    // lane l <-> dims 2l, 2l + 1 of every row; rows past the chunk re-read its last key
    const bool own = 2 * lane < head_dim;
    const int vl = own ? lane : 0;
    const uint32_t* vbase = reinterpret_cast<const uint32_t*>(Vc + static_cast<size_t>(kvh) * head_dim);  // uniform
    const size_t vrow = row / 2;  // in f16 pairs
    uint32_t vv[kAttnChunk];
    // in the kRope launch the new key's value comes from v_new and rows past the chunk's keys are
    // replaced by zeros below, so the loads stay below the new key's row where it is in this chunk
    const int vlast = j_new > 0 ? j_new - 1 : max(n - 1, 0);
#pragma unroll
    for (int j = 0; j < kAttnChunk; ++j) vv[j] = (vbase + static_cast<size_t>(s0 + min(j, vlast)) * vrow)[vl];
    __shared__ __align__(16) _Float16 rot[4][2][2 * kMaxPairs];  // [wave][q, k_new][dim]
    if constexpr (kRope) {
        // lane p rotates pair p (dims 2p, 2p + 1, or p, p + head_dim / 2) of the query and of the
        // new key, as rope_kernel does
        if (lane < pairs) {
            const float cs = dr.cs[lane], sn = dr.sn[lane];
            const int i0 = dr.neox ? lane : 2 * lane, i1 = dr.neox ? lane + pairs : 2 * lane + 1;
            const _Float16* qs = Q + (static_cast<size_t>(m) * heads + h) * head_dim;
            const _Float16* ks = dr.k_new + static_cast<size_t>(kvh) * head_dim;
            float a = static_cast<float>(qs[i0]), b = static_cast<float>(qs[i1]);
            rot[wl][0][i0] = static_cast<_Float16>(a * cs - b * sn);
            rot[wl][0][i1] = static_cast<_Float16>(a * sn + b * cs);
            a = static_cast<float>(ks[i0]);
            b = static_cast<float>(ks[i1]);
            const _Float16 k0 = static_cast<_Float16>(a * cs - b * sn), k1 = static_cast<_Float16>(a * sn + b * cs);
            rot[wl][1][i0] = k0;
            rot[wl][1][i1] = k1;
            if (j_new >= 0 && h % (heads / kv_heads) == 0) {  // one writer per KV head
                const size_t crow = static_cast<size_t>(pos) * row + static_cast<size_t>(kvh) * head_dim;
                dr.kc[crow + i0] = k0;
                dr.kc[crow + i1] = k1;
                const _Float16* vs = dr.v_new + static_cast<size_t>(kvh) * head_dim;
                dr.vc[crow + i0] = vs[i0];
                dr.vc[crow + i1] = vs[i1];
            }
        }
        // only this wave reads its LDS rows, and a wave's LDS operations complete in order
        __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        qp = reinterpret_cast<const uint32_t*>(rot[wl][0]);
    }
    if constexpr (kRope) {
        if (lane == j_new) {
            const u32x4* kn = reinterpret_cast<const u32x4*>(rot[wl][1]);
#pragma unroll
            for (int i = 0; i < kMaxPairs / 4; ++i)
                if (4 * i < pairs) kv[i] = kn[i];
        }
    }
    if constexpr (kRope) {
        const uint32_t vn = own ? reinterpret_cast<const uint32_t*>(dr.v_new + static_cast<size_t>(kvh) * head_dim)[lane] : 0u;
#pragma unroll
        for (int j = 0; j < kAttnChunk; ++j) vv[j] = j == j_new ? vn : (j < n ? vv[j] : 0u);
    }
    float dot = 0.0f;
#pragma unroll
    for (int i = 0; i < kMaxPairs / 4; ++i) {
        if (4 * i < pairs) {
            const uint32_t w[4] = {kv[i].x, kv[i].y, kv[i].z, kv[i].w};
#pragma unroll
            for (int e = 0; e < 4; ++e) dot = dot2(qp[4 * i + e], w[e], dot);
        }
    }
    const float sc = lane < n ? dot * scale : -INFINITY;
    float mx = sc;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    const float e = n > 0 ? expf(sc - mx) : 0.0f;  // 0 on masked lanes
    const float sum = wave_sum(e);

    // output: lane l <-> dims 2l, 2l + 1
    float acc0 = 0.0f, acc1 = 0.0f;
#pragma unroll
    for (int j = 0; j < kAttnChunk; ++j) {
        // lane j's weight, read into a scalar register (0 beyond the chunk's keys)
        const float pj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(e), j));
        h2v v;
        __builtin_memcpy(&v, &vv[j], 4);
        acc0 += pj * static_cast<float>(v[0]);
        acc1 += pj * static_cast<float>(v[1]);
    }
    if (chunks == 1) {
        if (own) {
            const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;
            _Float16* op = out + (static_cast<size_t>(m) * heads + h) * head_dim + 2 * lane;
            op[0] = static_cast<_Float16>(acc0 * inv);
            op[1] = static_cast<_Float16>(acc1 * inv);
        }
        return;
    }
    float* pp = part + static_cast<size_t>(wave) * (head_dim + 2);
    if (lane == 0) {
        pp[0] = n > 0 ? mx : -INFINITY;
        pp[1] = sum;
    }
    if (own) {
        pp[2 + 2 * lane] = acc0;
        pp[3 + 2 * lane] = acc1;
    }
}

// Merges the chunks of each (m, h) in chunk order.  One thread per output element.
__global__ __launch_bounds__(256) void attention_combine_kernel(const float* __restrict__ part, _Float16* __restrict__ out,
                                                              int q_len, int heads, int head_dim, int chunks) {
    const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int64_t total = static_cast<int64_t>(q_len) * heads * head_dim;
    if (idx >= total) return;
    const int d = static_cast<int>(idx % head_dim);
    const int64_t mh = idx / head_dim;
    const int h = static_cast<int>(mh % heads);
    const int m = static_cast<int>(mh / heads);
    const size_t stride = static_cast<size_t>(head_dim) + 2;
    auto at = [&](int c) { return part + ((static_cast<size_t>(m) * chunks + c) * heads + h) * stride; };
    // chunks are taken 8 at a time with all their loads issued first; the arithmetic runs in chunk
    // order
    constexpr int kG = 8;
    float mx = -INFINITY;
    for (int c0 = 0; c0 < chunks; c0 += kG) {
        float v[kG];
#pragma unroll
        for (int i = 0; i < kG; ++i) v[i] = c0 + i < chunks ? at(c0 + i)[0] : -INFINITY;
#pragma unroll
        for (int i = 0; i < kG; ++i) mx = fmaxf(mx, v[i]);
    }
    float sum = 0.0f, acc = 0.0f;
    for (int c0 = 0; c0 < chunks; c0 += kG) {
        float pm[kG], ps[kG], po[kG];
#pragma unroll
        for (int i = 0; i < kG; ++i) {
            const bool ok = c0 + i < chunks;
            const float* p = at(ok ? c0 + i : 0);
            pm[i] = p[0];
            ps[i] = ok ? p[1] : 0.0f;
            po[i] = p[2 + d];
        }
#pragma unroll
        for (int i = 0; i < kG; ++i) {
            if (ps[i] > 0.0f) {
                const float a = expf(pm[i] - mx);
                sum += ps[i] * a;
                acc += po[i] * a;
            }
        }
    }
    out[idx] = static_cast<_Float16>(sum > 0.0f ? acc / sum : 0.0f);
}

// Copies the call's new keys and values into their cache rows (one launch for both; two runtime copies
// took 4.9 us each).  vec: 16-byte pieces, else f16 values.
__global__ __launch_bounds__(256) void kv_append_kernel(const _Float16* __restrict__ k, const _Float16* __restrict__ v,
                                                      _Float16* __restrict__ kc, _Float16* __restrict__ vc, int64_t n, int vec) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    if (vec) {
        const u32x4 a = reinterpret_cast<const u32x4*>(k)[i], b = reinterpret_cast<const u32x4*>(v)[i];
        reinterpret_cast<u32x4*>(kc)[i] = a;
        reinterpret_cast<u32x4*>(vc)[i] = b;
    } else {
        kc[i] = k[i];
        vc[i] = v[i];
    }
}

// ---- KV cache pool (one per device) ----------------------------------------------------------
struct KvPool {
    _Float16* k = nullptr;
    _Float16* v = nullptr;
    int layers = 0, max_seq = 0, kv_heads = 0, head_dim = 0;
    size_t cap = 0;
};
std::mutex g_kv_mutex;
std::unordered_map<int, KvPool> g_kv;

// ---- keys split over workgroups ----------------------------------------------------------------
// Both matrix-core kernels below may cut a row's keys into ranges of `kps` keys, one workgroup each.
// A range's partial result of row (pos, head) is its running maximum m (base 2), the sum l of its
// weights 2^(x - m) and the unnormalised output: `o` [split][pos][head][D] and `ml` [split][pos][head]
// floats.  Ranges past the keys that a row tile sees are neither run nor read.
struct AttnSplit {
    float* o;
    float2* ml;
    int splits, kps;
};
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Keys that the rows of a tile of `tile_rows` rows (row r of a KV head's group: position r / group)
// can see, r any row of the tile.
__device__ __forceinline__ int tile_keys(int r, int tile_rows, int group, int q_len, int kv_len, int start_pos, int causal) {
    if (!causal) return kv_len;
    const int last = min((r / tile_rows * tile_rows + tile_rows - 1) / group, q_len - 1);
    return min(kv_len, start_pos + last + 1);
}

// Merges the partial results of each row.  Latency-bound (a few KiB per row): D / 4 threads hold a row's
// output and `sg` such groups share its ranges, four of them requested at once, so that a decode step's
// few rows take one or two memory round trips whatever the context; the groups are added in order
// through LDS.  8B decode at context 4000: 13.0 us with one thread per output element, chunk after chunk.
template <int D>
__global__ __launch_bounds__(256) void attention_merge_kernel(AttnSplit sp, _Float16* __restrict__ out, int q_len, int kv_len,
                                                            int heads, int group, int start_pos, int causal, int tile_rows,
                                                            int sg) {
    constexpr int kT = D / 4, kSlots = 256 / kT;
    __shared__ f32x4 so[kSlots][kT];
    __shared__ float2 sml[kSlots];
    const int slot = threadIdx.x / kT, t = threadIdx.x % kT, gi = slot % sg;
    const int64_t rows = static_cast<int64_t>(q_len) * heads;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * (kSlots / sg) + slot / sg;
    float m = -INFINITY, l = 0.0f;
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    if (row < rows) {
        const int pos = static_cast<int>(row / heads), h = static_cast<int>(row % heads);
        const int n = tile_keys(pos * group + h % group, tile_rows, group, q_len, kv_len, start_pos, causal);
        const int nv = (n + sp.kps - 1) / sp.kps;
        for (int c0 = gi; c0 < nv; c0 += 4 * sg) {
            float2 pm[4];
            f32x4 po[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int c = c0 + i * sg;
                const size_t at = static_cast<size_t>(c < nv ? c : c0) * rows + row;
                pm[i] = sp.ml[at];
                po[i] = reinterpret_cast<const f32x4*>(sp.o + at * D)[t];
                if (c >= nv) pm[i] = float2{-INFINITY, 0.0f};
            }
            const float mn = fmaxf(fmaxf(fmaxf(pm[0].x, pm[1].x), fmaxf(pm[2].x, pm[3].x)), m);
            const float a = m == mn ? 1.0f : __builtin_amdgcn_exp2f(m - mn);
            l *= a;
            acc *= a;
            m = mn;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (c0 + i * sg < nv) {
                    // a range of which the row sees no key has l = 0 (and mn may still be -inf)
                    const float w = pm[i].y == 0.0f ? 0.0f : __builtin_amdgcn_exp2f(pm[i].x - mn);
                    l += pm[i].y * w;
                    acc += po[i] * w;
                }
            }
        }
    }
    if (sg > 1) {
        so[slot][t] = acc;
        if (t == 0) sml[slot] = float2{m, l};
        __syncthreads();
        if (gi != 0) return;
        for (int i = 1; i < sg; ++i) {
            const float2 o = sml[slot + i];
            if (o.x == -INFINITY && o.y == 0.0f) continue;  // a group without ranges
            const float mn = fmaxf(m, o.x);
            const float a = m == mn ? 1.0f : __builtin_amdgcn_exp2f(m - mn);
            const float b = __builtin_amdgcn_exp2f(o.x - mn);
            l = l * a + o.y * b;
            acc = acc * a + so[slot + i][t] * b;
            m = mn;
        }
    }
    if (row >= rows) return;
    _Float16 h4[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) h4[i] = static_cast<_Float16>(acc[i] / l);
    __builtin_memcpy(out + row * D + 4 * t, h4, 8);
}

// ---- few query rows on the matrix cores ---------------------------------------------------------
// Attention of up to 16 rows (positions x query heads of one KV head) against one KV head's keys: the
// decode step, short chunks, and query groups that do not divide the 128-row tile below.  Bound by
// reading K and V (each once per row tile, whatever the number of query heads) and by the latency of
// one pass.  A wave takes 32 keys at a time, no LDS on the way:
//   * S^T = K Q^T on v_mfma_f32_16x16x32_f16: lane (l, q) = (lane % 16, lane / 16) loads 16 bytes of
//     key l's row per 32 dims (4 lanes read 64 contiguous bytes) and receives the scores of row l
//     with keys 4q..4q+3 of each 16-key tile;
//   * those 8 keys are the k order of the second product's operand, so the weights go straight from
//     the score registers into O^T += V^T P^T; lane (l, q) loads dims D/16 l .. of its 8 keys' V rows
//     (16 lanes read one whole row) and v_perm transposes them in registers;
//   * weights enter as 2^10 p = hi + lo in f16, two products (the scale cancels against the sum): 22 bits for
//     p >= 2^-13 of the range's maximum, an absolute error of 2^-35 of it below, where lo is subnormal or 0.
// The 4 waves of a workgroup take every fourth 32-key block of its range and are merged through LDS in
// wave order.  8B decode at context 4000 (16 MB of keys and values): 7.8 us and 4.3 us of merge, against
// 12.2 us and 13.0 us with one wave per (query head, 64 keys) on the vector ALUs, which reads each
// row once per query head and leaves four times the partial results.
// With kRope (one query position, the decode step): Q, k_new and v_new are the projections before RoPE.
// The rotation runs on the operand registers; the new key (position start_pos) and its value are taken
// from k_new / v_new, and the workgroup of row tile 0 whose range ends with it writes both into the
// cache row, which no lane of the launch reads.
constexpr int kRowsTile = 16, kRowsKeys = 32, kRowsWaves = 4;

template <int D>
__device__ __forceinline__ void rotate_row(f16x8 (&f)[D / 32], const DecodeRope& dr, int q) {
    if (dr.neox) {
#pragma unroll
        for (int db = 0; db < D / 64; ++db)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int p = 32 * db + 8 * q + e;
                const float cs = dr.cs[p], sn = dr.sn[p];
                const float a = static_cast<float>(f[db][e]), b = static_cast<float>(f[db + D / 64][e]);
                f[db][e] = static_cast<_Float16>(a * cs - b * sn);
                f[db + D / 64][e] = static_cast<_Float16>(a * sn + b * cs);
            }
    } else {
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int p = 16 * db + 4 * q + e;
                const float cs = dr.cs[p], sn = dr.sn[p];
                const float a = static_cast<float>(f[db][2 * e]), b = static_cast<float>(f[db][2 * e + 1]);
                f[db][2 * e] = static_cast<_Float16>(a * cs - b * sn);
                f[db][2 * e + 1] = static_cast<_Float16>(a * sn + b * cs);
            }
    }
}

template <int D, bool kRope>
__global__ __launch_bounds__(64 * kRowsWaves) void attention_rows_kernel(
    const _Float16* __restrict__ Q, const _Float16* __restrict__ Kc, const _Float16* __restrict__ Vc, _Float16* __restrict__ out,
    AttnSplit sp, int q_len, int kv_len, int heads, int kv_heads, int start_pos, float scale_log2, int causal, int rtiles,
    DecodeRope dr) {
    constexpr int kVW = D / 32;  // dwords of a lane's V slice: dims D/16 l .. D/16 l + D/16 - 1
    constexpr float kPScale = 10.0f;
    const int group = heads / kv_heads;
    const int g = static_cast<int>(blockIdx.x % kv_heads);
    const int rest = static_cast<int>(blockIdx.x / kv_heads);
    const int rt = rest % rtiles, split = rest / rtiles;
    const int n_rows = q_len * group;
    const int n_keys = tile_keys(rt * kRowsTile, kRowsTile, group, q_len, kv_len, start_pos, causal);
    const int k_begin = split * sp.kps, k_end = min(n_keys, k_begin + sp.kps);
    if (k_begin >= n_keys) return;
    const int lane = threadIdx.x & 63, l = lane & 15, q = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = min(rt * kRowsTile + l, n_rows - 1);  // rows past the last repeat it
    const int pos = r / group, head = g * group + r % group;
    const int row_end = causal ? min(kv_len, start_pos + pos + 1) : kv_len;  // keys this row sees
    const int vis_all = causal ? min(kv_len, start_pos + rt * kRowsTile / group + 1) : kv_len;  // keys every row sees
    const size_t kv_row = static_cast<size_t>(kv_heads) * D;
    const _Float16* kbase = Kc + static_cast<size_t>(g) * D;
    const _Float16* vbase = Vc + static_cast<size_t>(g) * D;

    f16x8 qf[D / 32];
    {
        const _Float16* qrow = Q + (static_cast<size_t>(pos) * heads + head) * D + 8 * q;
#pragma unroll
        for (int db = 0; db < D / 32; ++db) qf[db] = *reinterpret_cast<const f16x8*>(qrow + 32 * db);
        if constexpr (kRope) rotate_row<D>(qf, dr, q);
    }
    f32x4 o[D / 16];
    float m_run, l_run;
    // One pass over the wave's keys.  kCareful: the products run row by row, with the values that the row does
    // not see cleared and infinite or NaN ones weighted by p > 0 alone.
    auto scan = [&](auto careful) {
        constexpr bool kCareful = decltype(careful)::value;
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt) o[dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        m_run = -INFINITY;
        l_run = 0.0f;
        for (int kb = k_begin + kRowsKeys * w; kb < k_end; kb += kRowsKeys * kRowsWaves) {
            // keys past the tile's last read that key; their weights are zero
            f16x8 kf[2][D / 32];
            uint32_t vd[8][kVW];  // V slices of keys kb + 16 (j / 4) + 4 q + j % 4
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
                const int k = min(kb + 16 * tt + l, n_keys - 1);
                const _Float16* kr = kbase + static_cast<size_t>(k) * kv_row + 8 * q;
                if constexpr (kRope)
                    if (k == start_pos) kr = dr.k_new + static_cast<size_t>(g) * D + 8 * q;
#pragma unroll
                for (int db = 0; db < D / 32; ++db) kf[tt][db] = *reinterpret_cast<const f16x8*>(kr + 32 * db);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int k = min(kb + 16 * (j >> 2) + 4 * q + (j & 3), n_keys - 1);
                const _Float16* vr = vbase + static_cast<size_t>(k) * kv_row;
                if constexpr (kRope)
                    if (k == start_pos) vr = dr.v_new + static_cast<size_t>(g) * D;
                __builtin_memcpy(vd[j], __builtin_assume_aligned(vr + D / 16 * l, D / 8), 4 * kVW);
            }
            __builtin_amdgcn_sched_barrier(0);  // every load of the block is out before its first product
            if constexpr (kRope) {
                if (kb + kRowsKeys > start_pos) {  // the block with the new key
#pragma unroll
                    for (int tt = 0; tt < 2; ++tt) {
                        const bool is_new = min(kb + 16 * tt + l, n_keys - 1) == start_pos;
                        f16x8 rot[D / 32];
#pragma unroll
                        for (int db = 0; db < D / 32; ++db) rot[db] = kf[tt][db];
                        rotate_row<D>(rot, dr, q);
#pragma unroll
                        for (int db = 0; db < D / 32; ++db) kf[tt][db] = is_new ? rot[db] : kf[tt][db];
                        if (rt == 0 && kb + 16 * tt + l == start_pos) {
                            _Float16* kw = dr.kc + static_cast<size_t>(start_pos) * kv_row + static_cast<size_t>(g) * D + 8 * q;
#pragma unroll
                            for (int db = 0; db < D / 32; ++db) *reinterpret_cast<f16x8*>(kw + 32 * db) = rot[db];
                        }
                    }
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        if (rt == 0 && kb + 16 * (j >> 2) + 4 * q + (j & 3) == start_pos) {
                            _Float16* vw = dr.vc + static_cast<size_t>(start_pos) * kv_row + static_cast<size_t>(g) * D + D / 16 * l;
                            __builtin_memcpy(__builtin_assume_aligned(vw, D / 8), vd[j], 4 * kVW);
                        }
                }
            }
            // scores: x[4 tt + v] of key kb + 16 tt + 4 q + v
            const bool full = kb + kRowsKeys <= vis_all;
            float x[8];
            float mx = -INFINITY;
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
                f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int db = 0; db < D / 32; ++db) s = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[tt][db], qf[db], s, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    float y = s[v] * scale_log2;
                    if (!full && kb + 16 * tt + 4 * q + v >= row_end) y = -INFINITY;
                    x[4 * tt + v] = y;
                    mx = fmaxf(mx, y);
                }
            }
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            // a row that sees no key of this block keeps its state (its maximum may still be -inf)
            const bool sees = kb < row_end;
            const float m_new = sees ? fmaxf(m_run, mx) : m_run;
            const float corr = sees ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.0f;
            const float base = sees ? m_new - kPScale : 0.0f;
            float sum = 0.0f;
            f16x8 ph, pl, pw;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float p = __builtin_amdgcn_exp2f(x[i] - base);
                sum += p;
                ph[i] = static_cast<_Float16>(p);
                pl[i] = static_cast<_Float16>(p - static_cast<float>(ph[i]));
                if constexpr (kCareful) pw[i] = static_cast<_Float16>(p > 0.0f ? 1.0f : 0.0f);
            }
            sum += __shfl_xor(sum, 16, 64);
            sum += __shfl_xor(sum, 32, 64);
            l_run = l_run * corr + sum;
            m_run = m_new;
#pragma unroll
            for (int dt = 0; dt < D / 16; ++dt) o[dt] *= corr;
            // product dt: operand row l is dim D/16 l + dt of the lane's 8 keys
            __builtin_amdgcn_sched_barrier(0);  // and V's transposition waits for V alone
            if constexpr (!kCareful) {
#pragma unroll
                for (int dt = 0; dt < D / 16; ++dt) {
                    uint32_t t[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        t[i] = __builtin_amdgcn_perm(vd[2 * i + 1][dt >> 1], vd[2 * i][dt >> 1], (dt & 1) ? 0x07060302u : 0x05040100u);
                    f16x8 vf;
                    __builtin_memcpy(&vf, t, 16);
                    o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, ph, o[dt], 0, 0, 0);
                    o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pl, o[dt], 0, 0, 0);
                }
            } else {
#pragma unroll 1
                for (int rr = 0; rr < kRowsTile; ++rr) {
                    const int end = __shfl(row_end, rr, 64);
#pragma unroll
                    for (int dt = 0; dt < D / 16; ++dt) {
                        uint32_t fin[4], inf[4];  // the row's finite values, the others
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            uint32_t u = __builtin_amdgcn_perm(vd[2 * i + 1][dt >> 1], vd[2 * i][dt >> 1], (dt & 1) ? 0x07060302u : 0x05040100u);
                            const int k = kb + 16 * (i >> 1) + 4 * q + 2 * (i & 1);  // keys k, k + 1
                            u &= (k < end ? 0xFFFFu : 0u) | (k + 1 < end ? 0xFFFF0000u : 0u);
                            const uint32_t keep = ((u & 0x7C00u) != 0x7C00u ? 0xFFFFu : 0u) | ((u & 0x7C000000u) != 0x7C000000u ? 0xFFFF0000u : 0u);
                            fin[i] = u & keep;
                            inf[i] = u & ~keep;
                        }
                        f16x8 vf, vi;
                        __builtin_memcpy(&vf, fin, 16);
                        __builtin_memcpy(&vi, inf, 16);
                        f32x4 t = o[dt];
                        t = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, ph, t, 0, 0, 0);
                        t = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, pl, t, 0, 0, 0);
                        t = __builtin_amdgcn_mfma_f32_16x16x32_f16(vi, pw, t, 0, 0, 0);
                        o[dt] = l == rr ? t : o[dt];
                    }
                }
            }
        }
    };
    scan(std::false_type{});
    // An infinite or NaN value makes the plain products NaN where a row does not see it (0 weight) or where
    // its weight's lo term is 0 or negative: such a wave starts over, unless the scores themselves are NaN.
    bool bad = false;
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt)
#pragma unroll
        for (int v = 0; v < 4; ++v) bad |= o[dt][v] != o[dt][v];
    bad = bad && l_run == l_run;
    if (__builtin_expect(__ballot(bad) != 0, 0)) scan(std::true_type{});

    // Lane (l, q) holds dims D/4 q + D/16 v + dt of row l in o[dt][v].  Merge of the waves: LDS rows
    // padded by one 16-byte piece.
    constexpr int kRowF = D + 4;
    __shared__ __align__(16) float so[kRowsWaves][kRowsTile * kRowF];
    __shared__ float2 sml[kRowsWaves][kRowsTile];
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int dt = 0; dt < D / 16; dt += 4)
            *reinterpret_cast<f32x4*>(&so[w][l * kRowF + D / 4 * q + D / 16 * v + dt]) =
                f32x4{o[dt][v], o[dt + 1][v], o[dt + 2][v], o[dt + 3][v]};
    if (q == 0) sml[w][l] = float2{m_run, l_run};
    __syncthreads();
    constexpr int kPer = D / 16;  // dims per thread: 16 threads per row
    const int mr = threadIdx.x >> 4, d0 = kPer * (threadIdx.x & 15);
    const int row = rt * kRowsTile + mr;
    if (row >= n_rows) return;
    float mm = -INFINITY;
#pragma unroll
    for (int i = 0; i < kRowsWaves; ++i) mm = fmaxf(mm, sml[i][mr].x);
    float ls = 0.0f;
    f32x4 acc[kPer / 4];
#pragma unroll
    for (int j = 0; j < kPer / 4; ++j) acc[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < kRowsWaves; ++i) {
        const float2 ml = sml[i][mr];
        if (ml.x == -INFINITY && ml.y == 0.0f) continue;  // no key seen
        const float a = __builtin_amdgcn_exp2f(ml.x - mm);
        ls += ml.y * a;
#pragma unroll
        for (int j = 0; j < kPer / 4; ++j) acc[j] += *reinterpret_cast<const f32x4*>(&so[i][mr * kRowF + d0 + 4 * j]) * a;
    }
    const size_t orow = static_cast<size_t>(row / group) * heads + g * group + row % group;
    if (sp.splits == 1) {
        _Float16 hv[kPer];
#pragma unroll
        for (int j = 0; j < kPer; ++j) hv[j] = static_cast<_Float16>(acc[j / 4][j % 4] / ls);
        __builtin_memcpy(out + orow * D + d0, hv, 2 * kPer);
    } else {
        const size_t at = static_cast<size_t>(split) * q_len * heads + orow;
#pragma unroll
        for (int j = 0; j < kPer / 4; ++j) *reinterpret_cast<f32x4*>(sp.o + at * D + d0 + 4 * j) = acc[j];
        if (d0 == 0) sp.ml[at] = float2{mm, ls};
    }
}

// ---- prefill attention on the matrix cores --------------------------------------------------
// Flash-attention form for many query rows.  A workgroup of 4 waves owns 128 query rows: the
// 128 / G positions of a position tile times the G query heads of one KV head, which share every
// K and V row.  It walks the keys its rows can see in tiles of 64, staged through LDS
// (double-buffered, one barrier per tile):
//   * S = K Q^T on v_mfma_f32_32x32x16_f16.  A wave's 32 rows x 64 keys are two 32 x 32 tiles; K
//     fragments come from LDS, Q fragments stay in registers for the whole loop.  In an S tile a
//     lane holds one query row (lane mod 32) and 16 of the 32 keys, so the row's softmax
//     statistics need one exchange with the partner lane (lane ^ 32).
//   * fp32 online softmax in base 2 (2^(scale log2 e s - m), one fma per score; the row maximum is taken
//     over the raw scores, a negative scale moved to the query).  Bound by this vector work: 12000 causal
//     positions of 32 heads 1582 us with masks as selects and two products per score, 1398 us without.  Scaling
//     O only in tiles where some row's maximum grew was slower, as the branch keeps the products from
//     overlapping the exponentials: 40 positions over 3040 keys, unsplit, 92 us against 81 us; 100 positions
//     8.7 us against 8.2 us.
//   * O^T += V^T P^T on the same instruction.  P goes from the S registers into the B fragment
//     without leaving the lane: the k order of each 16-key block is the order the lane holds its
//     keys in.  V is staged transposed ([dim][key]) so an A fragment is two 8-byte LDS reads.
// Rows are divided by their softmax sum and rounded to fp16 once.  Position tiles run longest
// first (causal rows near the end see the most keys); with 8 KV heads the workgroups of one KV
// head land on one XCD and share its L2.
constexpr int kFaRows = 128, kFaKeys = 64, kFaThreads = 256;

template <int D>
struct FaGeom {
    static constexpr int kRowK = D + 8;                      // f16 per staged K row (16-byte pad)
    static constexpr int kRowV = kFaKeys + 4;                // f16 per staged V^T row (8-byte pad)
    static constexpr int kK = kFaKeys * kRowK;               // f16 per K buffer
    static constexpr int kV = D * kRowV;                     // f16 per V^T buffer
    static constexpr int kBuf = kK + kV;
    static constexpr size_t kLdsBytes = 2 * static_cast<size_t>(kBuf) * sizeof(_Float16);
    static constexpr int kChunks = D / 8;                    // 16-byte chunks per row
    static constexpr int kKUnits = kFaKeys * kChunks / kFaThreads;        // K chunks per thread
    static constexpr int kVUnits = (kFaKeys / 2) * kChunks / kFaThreads;  // V (key pair, chunk) per thread
    static_assert(kKUnits >= 1 && kVUnits >= 1, "head_dim 64 or 128");
};

extern __shared__ __align__(16) _Float16 fa_lds[];

template <int D>
__global__ __launch_bounds__(kFaThreads, 2) void attention_mfma_kernel(
    const _Float16* __restrict__ Q, const _Float16* __restrict__ Kc, const _Float16* __restrict__ Vc,
    _Float16* __restrict__ out, AttnSplit sp, int q_len, int kv_len, int heads, int kv_heads, int start_pos,
    float scale_log2, int causal, int ptiles) {
    using FG = FaGeom<D>;
    const int group = heads / kv_heads;
    const int ppw = kFaRows / group;  // positions per workgroup
    const int g = static_cast<int>(blockIdx.x % kv_heads);
    const int pt = ptiles - 1 - static_cast<int>(blockIdx.x / kv_heads) % ptiles;
    const int split = static_cast<int>(blockIdx.x / kv_heads) / ptiles;
    const int p0 = pt * ppw;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
    const int r = 32 * (tid >> 6) + l32;  // row of the workgroup
    const int pos = p0 + r / group;
    const int head = g * group + r % group;
    const int p_last = min(p0 + ppw, q_len) - 1;
    const int n_keys = causal ? min(kv_len, start_pos + p_last + 1) : kv_len;
    const int t0 = split * (sp.kps / kFaKeys);
    const int n_tiles = min((n_keys + kFaKeys - 1) / kFaKeys, t0 + sp.kps / kFaKeys);
    if (t0 >= n_tiles) return;
    const int vis_all = causal ? min(kv_len, start_pos + p0 + 1) : kv_len;    // keys every row sees
    const int row_end = causal ? min(kv_len, start_pos + pos + 1) : kv_len;   // keys this row sees
    const size_t kv_row = static_cast<size_t>(kv_heads) * D;
    const _Float16* kbase = Kc + static_cast<size_t>(g) * D;
    const _Float16* vbase = Vc + static_cast<size_t>(g) * D;

    // Q fragments of row (pos, head): dims 16 db + 8 h .. + 7 (rows past q_len read the last row)
    f16x8 qf[D / 16];
    {
        const _Float16* qrow = Q + (static_cast<size_t>(min(pos, q_len - 1)) * heads + head) * D + 8 * h;
#pragma unroll
        for (int db = 0; db < D / 16; ++db) __builtin_memcpy(&qf[db], qrow + 16 * db, 16);
        // a negative scale: the same scores from -q and its magnitude
        if (scale_log2 < 0.0f) {
#pragma unroll
            for (int db = 0; db < D / 16; ++db) qf[db] = -qf[db];
            scale_log2 = -scale_log2;
        }
    }

    // Staging of key tile t: thread units of K (key, chunk) and of V (key pair, chunk); keys past
    // kv_len read the last key (finite values, masked out of the softmax).
    u32x4 kr[FG::kKUnits], vr[FG::kVUnits][2];
    auto load = [&](int t) {
        const int kb = t * kFaKeys;
#pragma unroll
        for (int i = 0; i < FG::kKUnits; ++i) {
            const int u = tid + kFaThreads * i, key = u / FG::kChunks, c = u % FG::kChunks;
            const int k = min(kb + key, kv_len - 1);
            kr[i] = *reinterpret_cast<const u32x4*>(kbase + static_cast<size_t>(k) * kv_row + 8 * c);
        }
#pragma unroll
        for (int i = 0; i < FG::kVUnits; ++i) {
            const int u = tid + kFaThreads * i, kp = u % (kFaKeys / 2), c = u / (kFaKeys / 2);
            const int k0 = min(kb + 2 * kp, kv_len - 1), k1 = min(kb + 2 * kp + 1, kv_len - 1);
            vr[i][0] = *reinterpret_cast<const u32x4*>(vbase + static_cast<size_t>(k0) * kv_row + 8 * c);
            vr[i][1] = *reinterpret_cast<const u32x4*>(vbase + static_cast<size_t>(k1) * kv_row + 8 * c);
        }
    };
    auto store = [&](int buf) {
        _Float16* sk = fa_lds + buf * FG::kBuf;
        _Float16* sv = sk + FG::kK;
#pragma unroll
        for (int i = 0; i < FG::kKUnits; ++i) {
            const int u = tid + kFaThreads * i, key = u / FG::kChunks, c = u % FG::kChunks;
            *reinterpret_cast<u32x4*>(sk + key * FG::kRowK + 8 * c) = kr[i];
        }
#pragma unroll
        for (int i = 0; i < FG::kVUnits; ++i) {
            const int u = tid + kFaThreads * i, kp = u % (kFaKeys / 2), c = u / (kFaKeys / 2);
            // V^T[8c + e][2kp, 2kp + 1] = (V[k0][8c + e], V[k1][8c + e]); dword m of a row chunk
            // holds dims 2m, 2m + 1
            uint32_t* col = reinterpret_cast<uint32_t*>(sv + 8 * c * FG::kRowV + 2 * kp);
            const u32x4 a = vr[i][0], b = vr[i][1];
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                col[(2 * m) * (FG::kRowV / 2)] = __builtin_amdgcn_perm(b[m], a[m], 0x05040100u);
                col[(2 * m + 1) * (FG::kRowV / 2)] = __builtin_amdgcn_perm(b[m], a[m], 0x07060302u);
            }
        }
    };

    f32x16 o[D / 32];
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[dt][v] = 0.0f;
    float m_run = -INFINITY, l_run = 0.0f;

    // waves whose 32 rows all lie past q_len only stage
    const bool live = p0 + __builtin_amdgcn_readfirstlane(32 * (tid >> 6)) / group < q_len;
    load(t0);
    store(t0 & 1);
    __syncthreads();
    for (int t = t0; t < n_tiles; ++t) {
        if (t + 1 < n_tiles) load(t + 1);
        if (!live) {
            if (t + 1 < n_tiles) store((t + 1) & 1);
            __syncthreads();
            continue;
        }
        const _Float16* sk = fa_lds + (t & 1) * FG::kBuf;
        const _Float16* sv = sk + FG::kK;
        // S^T tiles: register v of tile tt is key 32 tt + 8 (v / 4) + 4 h + v % 4 of the row l32
        f32x16 s[2];
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
#pragma unroll
            for (int v = 0; v < 16; ++v) s[tt][v] = 0.0f;
#pragma unroll
            for (int db = 0; db < D / 16; ++db) {
                f16x8 kf;
                __builtin_memcpy(&kf, sk + (32 * tt + l32) * FG::kRowK + 16 * db + 8 * h, 16);
                s[tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[db], s[tt], 0, 0, 0);
            }
        }
        const int kb = t * kFaKeys;
        const bool full = kb + kFaKeys <= vis_all;
        // the masks are a branch of their own: as selects they cost every tile two instructions per score
        if (!full) {
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    if (kb + 32 * tt + 8 * (v >> 2) + 4 * h + (v & 3) >= row_end) s[tt][v] = -INFINITY;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int v = 0; v < 16; ++v) mx = fmaxf(mx, s[tt][v]);
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        // a row that sees no key of this tile keeps its state (its maximum may still be -inf)
        const bool sees = kb < row_end;
        const float m_new = sees ? fmaxf(m_run, mx * scale_log2) : m_run;
        const float corr = sees ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.0f;
        const float base = sees ? m_new : 0.0f;
        float sum = 0.0f;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float p = __builtin_amdgcn_exp2f(__fmaf_rn(s[tt][v], scale_log2, -base));
                s[tt][v] = p;
                sum += p;
            }
        sum += __shfl_xor(sum, 32, 64);
        l_run = l_run * corr + sum;
        m_run = m_new;
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
            for (int v = 0; v < 16; ++v) o[dt][v] *= corr;
        // 16-key block b: lane half h holds keys 16 b + 4 h + (0..3) and 16 b + 8 + 4 h + (0..3)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            f16x8 pf;
#pragma unroll
            for (int e = 0; e < 8; ++e) pf[e] = static_cast<_Float16>(s[b >> 1][8 * (b & 1) + e]);
#pragma unroll
            for (int dt = 0; dt < D / 32; ++dt) {
                const _Float16* vrow = sv + (32 * dt + l32) * FG::kRowV + 16 * b + 4 * h;
                f16x8 vf;
                __builtin_memcpy(&vf, vrow, 8);
                __builtin_memcpy(reinterpret_cast<char*>(&vf) + 8, vrow + 8, 8);
                o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pf, o[dt], 0, 0, 0);
            }
        }
        if (t + 1 < n_tiles) store((t + 1) & 1);
        __syncthreads();
    }

    if (pos >= q_len) return;
    if (sp.splits > 1) {
        const size_t at = (static_cast<size_t>(split) * q_len + pos) * heads + head;
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4)
                *reinterpret_cast<f32x4*>(sp.o + at * D + 32 * dt + 8 * q4 + 4 * h) =
                    f32x4{o[dt][4 * q4], o[dt][4 * q4 + 1], o[dt][4 * q4 + 2], o[dt][4 * q4 + 3]};
        if (h == 0) sp.ml[at] = float2{m_run, l_run};
    } else {
        const float inv = 1.0f / l_run;
        _Float16* orow = out + (static_cast<size_t>(pos) * heads + head) * D;
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                _Float16 v4[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) v4[i] = static_cast<_Float16>(o[dt][4 * q4 + i] * inv);
                __builtin_memcpy(orow + 32 * dt + 8 * q4 + 4 * h, v4, 8);
            }
    }
}

int attn_chunks(int kv_len) { return kv_len <= 0 ? 1 : (kv_len + kAttnChunk - 1) / kAttnChunk; }

// Which attention kernel serves a call, and how its keys are split over workgroups.
//   kMfma: >= kFaMinRows query positions (fewer leave the 128-row tile mostly empty) of a query group
//          that divides 128;
//   kRows: the other calls of head_dim 64 and 128;
//   kLanes: other head sizes, and Q / K / V that are not 16-byte aligned.
constexpr int kFaMinRows = 16;
// Workgroups that a split grid is cut to: two per CU, what the 128-row tile's LDS allows.  (The 16-row tile of
// head_dim 128 that rotates its query fits once per CU; its ranges past 256 run in a second round.)
constexpr int64_t kAttnFill = 512, kAttnCus = 256;
enum class AttnKind { kMfma, kRows, kLanes };
struct AttnPlan {
    AttnKind kind;
    int tile_rows, tiles;  // rows per tile (positions x query heads of a KV head), row tiles
    int splits, kps;       // key ranges per row tile and keys per range
    size_t bytes;          // workspace of the partial results
};

// Keys per range: the key blocks of all row tiles spread over kAttnFill workgroups (a block: 64 keys of
// the 128-row tile, at least two per range, or 32 keys of each wave of the 16-row tile).  A tile's keys
// are split only while the grid leaves half of the workgroups' places empty, and where that saves more
// than it costs:
//   saved  the longest tile's blocks, 1.6 / 1.0 us each in the 128-row tile (head_dim 128 / 64; 1.4 times
//          that with two workgroups on a CU) and 1.6 / 0.8 us in the 16-row tile;
//   cost   the merge, 4.5 us after the 128-row tile (launch gap and more ranges per CU) and 2.5 us after the
//          16-row tile, and the partial results, written and read at 5 TB/s.
// us, unsplit / split, 32 heads, 8 of keys, head_dim 128:
//   200 positions over 200 keys   9.8 / 14.9       400 keys  16.4 / 17.4    3200 keys  ~90 / 30
//   500 positions over 500 keys  18.1 / 25.0       700 keys  23.1 / 32.7    3500 keys  ~98 / 53.5
//   1000 positions over 1000 keys 31.8 / 35.6     1200 keys  36.5 / 44.5    4000 keys ~114 / 95
//   whole 8B decode layer         201 keys 46.5 / 47.5    401 keys 50.0 / 47.3    601 keys 52.6 / 48.6
// and 4 heads of 64: 40 positions over 240 keys 7.3 / 9.5, 3040 keys 52 / 10; 1B decode layer (32 heads of 64)
// 201 keys 45.3 / 47.9, 401 keys 47.2 / 47.6, 601 keys 48.3 / 48.1.
AttnPlan attn_plan(int q_len, int kv_len, int heads, int kv_heads, int head_dim, int start_pos, bool causal, bool aligned,
                   bool may_split) {
    const int group = heads / kv_heads;
    const int64_t rows = static_cast<int64_t>(q_len) * group;
    const size_t row_bytes = static_cast<size_t>(q_len) * heads * (head_dim + 2) * sizeof(float);
    AttnPlan p{};
    if ((head_dim != 64 && head_dim != 128) || kv_len <= 0 || !aligned || rows > (1 << 30)) {
        p.kind = AttnKind::kLanes;
        p.splits = attn_chunks(kv_len);
        p.kps = kAttnChunk;
        p.bytes = p.splits > 1 ? row_bytes * p.splits : 0;
        return p;
    }
    const bool mfma = q_len >= kFaMinRows && kFaRows % group == 0;
    p.kind = mfma ? AttnKind::kMfma : AttnKind::kRows;
    p.tile_rows = mfma ? kFaRows : kRowsTile;
    p.tiles = static_cast<int>((rows + p.tile_rows - 1) / p.tile_rows);
    const int block = mfma ? kFaKeys : kRowsKeys * kRowsWaves;
    const int64_t wgs = static_cast<int64_t>(p.tiles) * kv_heads;
    int64_t blocks = 0;  // of one KV head
    int most = 0;        // of one row tile
    for (int t = 0; t < p.tiles; ++t) {
        int n = kv_len;
        if (causal) {
            const int64_t last = std::min((static_cast<int64_t>(t + 1) * p.tile_rows - 1) / group, static_cast<int64_t>(q_len) - 1);
            n = static_cast<int>(std::min<int64_t>(kv_len, start_pos + last + 1));
        }
        const int b = (n + block - 1) / block;
        blocks += b;
        most = std::max(most, b);
    }
    int per = most;
    if (may_split && 2 * wgs <= kAttnFill) {
        const int64_t even = (blocks * kv_heads + kAttnFill - 1) / kAttnFill;
        const int max_splits = static_cast<int>(2 * kAttnFill / wgs);
        const int range = static_cast<int>(std::min<int64_t>(most, std::max<int64_t>({even, mfma ? 2 : 1, (most + max_splits - 1) / max_splits})));
        const double block_us = head_dim == 128 ? 1.6 : mfma ? 1.0 : 0.8;
        const double run = static_cast<double>(blocks) / range * kv_heads;  // workgroups that have keys
        const double part_bytes = static_cast<double>(row_bytes) * blocks / (static_cast<double>(range) * p.tiles);
        const double saved = block_us * (most - range * (mfma && run > kAttnCus ? 1.4 : 1.0));
        if (saved > (mfma ? 4.5 : 2.5) + 2.0 * part_bytes / 5e6) per = range;
    }
    p.splits = (most + per - 1) / per;
    p.kps = per * block;
    // Room for any call of as many rows and keys or fewer: at most a partial result per row and block, and
    // (max_splits) 2 kAttnFill row tiles of them.  The plan's own need goes up and down with the context (8192
    // keys make 64 ranges, 8193 make 33), so a buffer sized by it would grow, and move, after a longer call.
    if (may_split && kv_len > block)
        p.bytes = static_cast<size_t>(std::min<int64_t>(static_cast<int64_t>(q_len) * heads * ((kv_len + block - 1) / block),
                                                        2 * kAttnFill * p.tile_rows)) * (head_dim + 2) * sizeof(float);
    return p;
}

AttnSplit attn_split(const AttnPlan& p, void* part, int q_len, int heads, int head_dim) {
    AttnSplit sp{};
    sp.splits = p.splits;
    sp.kps = p.kps;
    sp.o = static_cast<float*>(part);
    if (p.splits > 1) sp.ml = reinterpret_cast<float2*>(sp.o + static_cast<size_t>(p.splits) * q_len * heads * head_dim);
    return sp;
}

bool attn_aligned(const void* Q, const void* K, const void* V) {
    return (reinterpret_cast<uintptr_t>(Q) | reinterpret_cast<uintptr_t>(K) | reinterpret_cast<uintptr_t>(V)) % 16 == 0;
}

}  // namespace

// ---- launchers (validated arguments) --------------------------------------------------------
hipError_t launch_rmsnorm(const void* x, const void* res, const void* w, int w_f32, void* h_out, void* out, int M, int K,
                          float eps, hipStream_t stream) {
    if (M <= 0 || K <= 0) return hipSuccess;
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(M), dim3(kNormThreads), 0, stream, static_cast<const _Float16*>(x),
                           static_cast<const _Float16*>(res), w, w_f32, static_cast<_Float16*>(h_out), static_cast<_Float16*>(out), K, eps);
    };
    if (K % 8 != 0 || K > 2048 * 8) go(rmsnorm_kernel);
    else if (K <= 2048 * 2) go(rmsnorm_reg_kernel<2>);
    else if (K <= 2048 * 4) go(rmsnorm_reg_kernel<4>);
    else go(rmsnorm_reg_kernel<8>);
    return hipGetLastError();
}

hipError_t launch_residual_add(const void* x, const void* r, void* out, int64_t n, hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    const int64_t items = (n & 7) == 0 ? n / 8 : n;
    hipLaunchKernelGGL(residual_add_kernel, dim3(static_cast<unsigned>((items + 255) / 256)), dim3(256), 0, stream,
                       static_cast<const _Float16*>(x), static_cast<const _Float16*>(r), static_cast<_Float16*>(out), n);
    return hipGetLastError();
}

hipError_t launch_bias_add(void* y, const void* b, int rows, int n, hipStream_t stream) {
    const int64_t total = static_cast<int64_t>(rows) * n;
    const int blocks = static_cast<int>(std::min<int64_t>((total + 255) / 256, 4096));
    hipLaunchKernelGGL(bias_add_kernel, dim3(blocks), dim3(256), 0, stream, static_cast<_Float16*>(y),
                       static_cast<const _Float16*>(b), n, total);
    return hipGetLastError();
}

hipError_t launch_swiglu(const void* g, const void* u, void* out, int64_t n, hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    const int64_t items = (n & 7) == 0 ? n / 8 : n;
    hipLaunchKernelGGL(swiglu_kernel, dim3(static_cast<unsigned>((items + 255) / 256)), dim3(256), 0, stream,
                       static_cast<const _Float16*>(g), static_cast<const _Float16*>(u), static_cast<_Float16*>(out), n);
    return hipGetLastError();
}

hipError_t launch_rope(const void* q, void* q_out, int n_q, const void* k, void* k_out, const void* v, void* v_out, int n_k,
                       int seq_len, int head_dim, int pos_offset, float freq_base, bool neox, hipStream_t stream) {
    if (seq_len <= 0 || n_q + n_k <= 0) return hipSuccess;
    RopeFreq fr;
    for (int i = 0; i < head_dim / 2; ++i)
        fr.inv[i] = 1.0f / std::pow(freq_base, static_cast<float>(2 * i) / static_cast<float>(head_dim));
    // heads per block: as many as leave about 2048 blocks, at least one pass of the block's threads
    const int heads = n_q + n_k, groups = 256 / (head_dim / 2);  // rotated heads that a block holds at a time
    const int hg = std::min(groups, heads), ppb = groups / hg;
    const int64_t want = (static_cast<int64_t>(heads) * seq_len + 2047) / 2048;
    const int hpb = static_cast<int>(std::min<int64_t>(heads, std::max<int64_t>(want, hg)));
    hipLaunchKernelGGL(rope_kernel, dim3(static_cast<unsigned>((seq_len + ppb - 1) / ppb), static_cast<unsigned>((heads + hpb - 1) / hpb)),
                       dim3(256), 0, stream,
                       static_cast<const _Float16*>(q), static_cast<_Float16*>(q_out), n_q, static_cast<const _Float16*>(k),
                       static_cast<_Float16*>(k_out), static_cast<const _Float16*>(v), static_cast<_Float16*>(v_out), n_k,
                       seq_len, head_dim, pos_offset, neox ? 1 : 0, hpb, hg, ppb, fr);
    return hipGetLastError();
}

size_t attention_workspace_bytes(const void* Q, const void* K, const void* V, int q_len, int kv_len, int heads,
                                 int kv_heads, int head_dim, int start_pos, bool causal, bool may_split) {
    const bool al = attn_aligned(Q, K, V);
    const AttnPlan p = attn_plan(q_len, kv_len, heads, kv_heads, head_dim, std::min(start_pos, kv_len), causal, al, may_split);
    return p.bytes;
}

namespace {

hipError_t launch_merge(const AttnPlan& p, const AttnSplit& sp, _Float16* out, int q_len, int kv_len, int heads, int kv_heads,
                        int head_dim, int start_pos, bool causal, hipStream_t stream) {
    const int64_t rows = static_cast<int64_t>(q_len) * heads;
    const int slots = 1024 / head_dim;
    int sg = 1;  // groups of threads per row: four ranges each, as long as the rows leave CUs idle
    while (sg < slots && 4 * sg < p.splits && rows * sg < 8192) sg *= 2;
    const int64_t blocks = (rows * sg + slots - 1) / slots;
    auto go = [&](auto dc) {
        hipLaunchKernelGGL((attention_merge_kernel<decltype(dc)::value>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, sp,
                           out, q_len, kv_len, heads, heads / kv_heads, start_pos, causal ? 1 : 0, p.tile_rows, sg);
    };
    if (head_dim == 128) go(std::integral_constant<int, 128>{});
    else go(std::integral_constant<int, 64>{});
    return hipGetLastError();
}

template <int D>
hipError_t launch_attention_mfma(const AttnPlan& p, const AttnSplit& sp, const void* Q, const void* K, const void* V, void* out,
                                 int q_len, int kv_len, int heads, int kv_heads, int start_pos, float scale, bool causal,
                                 hipStream_t stream) {
    using FG = FaGeom<D>;
    static std::once_flag once;
    static hipError_t attr = hipSuccess;
    std::call_once(once, [] {
        attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&attention_mfma_kernel<D>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(FG::kLdsBytes));
    });
    if (attr != hipSuccess) return attr;
    const float scale_log2 = scale * 1.4426950408889634f;
    hipLaunchKernelGGL((attention_mfma_kernel<D>), dim3(static_cast<unsigned>(p.tiles * kv_heads * p.splits)), dim3(kFaThreads),
                       FG::kLdsBytes, stream, static_cast<const _Float16*>(Q), static_cast<const _Float16*>(K),
                       static_cast<const _Float16*>(V), static_cast<_Float16*>(out), sp, q_len, kv_len, heads, kv_heads,
                       start_pos, scale_log2, causal ? 1 : 0, p.tiles);
    return hipGetLastError();
}

template <int D, bool kRope>
hipError_t launch_attention_rows(const AttnPlan& p, const AttnSplit& sp, const void* Q, const void* K, const void* V, void* out,
                                 int q_len, int kv_len, int heads, int kv_heads, int start_pos, float scale, bool causal,
                                 const DecodeRope& dr, hipStream_t stream) {
    const int64_t blocks = static_cast<int64_t>(p.tiles) * kv_heads * p.splits;
    if (blocks > INT32_MAX) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL((attention_rows_kernel<D, kRope>), dim3(static_cast<unsigned>(blocks)), dim3(64 * kRowsWaves), 0, stream,
                       static_cast<const _Float16*>(Q), static_cast<const _Float16*>(K), static_cast<const _Float16*>(V),
                       static_cast<_Float16*>(out), sp, q_len, kv_len, heads, kv_heads, start_pos,
                       scale * 1.4426950408889634f, causal ? 1 : 0, p.tiles, dr);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_kv_append(const void* k, const void* v, void* kc, void* vc, int64_t n, hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    const uintptr_t al = reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) | reinterpret_cast<uintptr_t>(kc) |
                         reinterpret_cast<uintptr_t>(vc);
    const bool vec = al % 16 == 0 && n % 8 == 0;
    const int64_t items = vec ? n / 8 : n;
    hipLaunchKernelGGL(kv_append_kernel, dim3(static_cast<unsigned>((items + 255) / 256)), dim3(256), 0, stream,
                       static_cast<const _Float16*>(k), static_cast<const _Float16*>(v), static_cast<_Float16*>(kc),
                       static_cast<_Float16*>(vc), items, vec ? 1 : 0);
    return hipGetLastError();
}

hipError_t launch_attention(const void* Q, const void* K, const void* V, void* out, void* part, int q_len, int kv_len,
                            int heads, int kv_heads, int head_dim, int start_pos, float scale, bool causal, bool may_split,
                            hipStream_t stream) {
    if (q_len <= 0 || heads <= 0) return hipSuccess;
    const bool aligned = attn_aligned(Q, K, V);
    start_pos = std::min(start_pos, kv_len);  // every row sees all keys from there on
    const AttnPlan p = attn_plan(q_len, kv_len, heads, kv_heads, head_dim, start_pos, causal, aligned, may_split);
    hipError_t e;
    if (p.kind != AttnKind::kLanes) {
        const AttnSplit sp = attn_split(p, part, q_len, heads, head_dim);
        auto go = [&](auto dc) {
            constexpr int D = decltype(dc)::value;
            return p.kind == AttnKind::kMfma
                       ? launch_attention_mfma<D>(p, sp, Q, K, V, out, q_len, kv_len, heads, kv_heads, start_pos, scale, causal, stream)
                       : launch_attention_rows<D, false>(p, sp, Q, K, V, out, q_len, kv_len, heads, kv_heads, start_pos, scale,
                                                         causal, DecodeRope{}, stream);
        };
        e = head_dim == 128 ? go(std::integral_constant<int, 128>{}) : go(std::integral_constant<int, 64>{});
        if (e != hipSuccess || p.splits == 1) return e;
        return launch_merge(p, sp, static_cast<_Float16*>(out), q_len, kv_len, heads, kv_heads, head_dim, start_pos, causal, stream);
    }
    const int chunks = attn_chunks(kv_len);
    const int64_t waves = static_cast<int64_t>(q_len) * heads * chunks;
    const dim3 grid(static_cast<unsigned>((waves + 3) / 4));
    auto go = [&](auto dc) {
        constexpr int D = decltype(dc)::value;
        hipLaunchKernelGGL((attention_kernel<D>), grid, dim3(256), 0, stream, static_cast<const _Float16*>(Q),
                           static_cast<const _Float16*>(K), static_cast<const _Float16*>(V), static_cast<_Float16*>(out),
                           static_cast<float*>(part), q_len, kv_len, heads, kv_heads, head_dim, start_pos, scale,
                           causal ? 1 : 0, chunks);
    };
    if (head_dim % 8 == 0 && head_dim <= 128 && aligned)
        hipLaunchKernelGGL((attention_keys_kernel<false>), grid, dim3(256), 0, stream, static_cast<const _Float16*>(Q),
                           static_cast<const _Float16*>(K), static_cast<const _Float16*>(V), static_cast<_Float16*>(out),
                           static_cast<float*>(part), q_len, kv_len, heads, kv_heads, head_dim, start_pos, scale,
                           causal ? 1 : 0, chunks, DecodeRope{});
    else if (head_dim <= 64) go(std::integral_constant<int, 1>{});
    else if (head_dim <= 128) go(std::integral_constant<int, 2>{});
    else go(std::integral_constant<int, 4>{});
    e = hipGetLastError();
    if (e != hipSuccess || chunks == 1) return e;
    const int64_t n = static_cast<int64_t>(q_len) * heads * head_dim;
    hipLaunchKernelGGL(attention_combine_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, stream,
                       static_cast<const float*>(part), static_cast<_Float16*>(out), q_len, heads, head_dim, chunks);
    return hipGetLastError();
}

hipError_t launch_attention_decode_rope(const void* q, const void* k_new, const void* v_new, void* kc, void* vc, void* out,
                                        void* part, int kv_len, int heads, int kv_heads, int head_dim, float scale,
                                        float freq_base, bool neox, hipStream_t stream) {
    const uintptr_t al = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k_new) |
                         reinterpret_cast<uintptr_t>(v_new) | reinterpret_cast<uintptr_t>(kc) | reinterpret_cast<uintptr_t>(vc);
    if (kv_len <= 0 || heads <= 0 || head_dim % 8 != 0 || head_dim > 128 || (al & 15u) != 0) return hipErrorNotSupported;
    DecodeRope dr{};
    dr.k_new = static_cast<const _Float16*>(k_new);
    dr.v_new = static_cast<const _Float16*>(v_new);
    dr.kc = static_cast<_Float16*>(kc);
    dr.vc = static_cast<_Float16*>(vc);
    dr.neox = neox ? 1 : 0;
    // the angle as the RoPE kernel forms it (fp32 position x fp32 inverse frequency); its cosine
    // and sine evaluated here once for the step
    for (int i = 0; i < head_dim / 2; ++i) {
        const float inv = 1.0f / std::pow(freq_base, static_cast<float>(2 * i) / static_cast<float>(head_dim));
        const float ang = static_cast<float>(kv_len - 1) * inv;
        dr.cs[i] = static_cast<float>(std::cos(static_cast<double>(ang)));
        dr.sn[i] = static_cast<float>(std::sin(static_cast<double>(ang)));
    }
    const AttnPlan p = attn_plan(1, kv_len, heads, kv_heads, head_dim, kv_len - 1, true, true, true);
    if (p.kind == AttnKind::kRows) {
        const AttnSplit sp = attn_split(p, part, 1, heads, head_dim);
        const hipError_t e = head_dim == 128 ? launch_attention_rows<128, true>(p, sp, q, kc, vc, out, 1, kv_len, heads, kv_heads,
                                                                                kv_len - 1, scale, true, dr, stream)
                                             : launch_attention_rows<64, true>(p, sp, q, kc, vc, out, 1, kv_len, heads, kv_heads,
                                                                               kv_len - 1, scale, true, dr, stream);
        if (e != hipSuccess || p.splits == 1) return e;
        return launch_merge(p, sp, static_cast<_Float16*>(out), 1, kv_len, heads, kv_heads, head_dim, kv_len - 1, true, stream);
    }
    const int chunks = p.splits;
    const int64_t waves = static_cast<int64_t>(heads) * chunks;
    hipLaunchKernelGGL((attention_keys_kernel<true>), dim3(static_cast<unsigned>((waves + 3) / 4)), dim3(256), 0, stream,
                       static_cast<const _Float16*>(q), static_cast<const _Float16*>(kc), static_cast<const _Float16*>(vc),
                       static_cast<_Float16*>(out), static_cast<float*>(part), 1, kv_len, heads, kv_heads, head_dim,
                       kv_len - 1, scale, 1, chunks, dr);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || chunks == 1) return e;
    const int64_t n = static_cast<int64_t>(heads) * head_dim;
    hipLaunchKernelGGL(attention_combine_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, stream,
                       static_cast<const float*>(part), static_cast<_Float16*>(out), 1, heads, head_dim, chunks);
    return hipGetLastError();
}

// ---- KV cache pool ----------------------------------------------------------------------------
LayerStatus kv_cache_init(int layers, int max_seq, int kv_heads, int head_dim) {
    if (layers <= 0 || max_seq <= 0 || kv_heads <= 0 || head_dim <= 0)
        return {QMM_ERR_INVALID_ARGUMENT, "KV cache dimensions must all be positive."};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return {QMM_ERR_HIP, std::string("hipGetDevice: ") + hipGetErrorString(e)};
    std::lock_guard<std::mutex> lock(g_kv_mutex);
    KvPool& p = g_kv[dev];
    const size_t need = static_cast<size_t>(layers) * max_seq * kv_heads * head_dim * sizeof(_Float16);
    if (need > p.cap) {
        if (p.k) (void)hipFree(p.k);
        if (p.v) (void)hipFree(p.v);
        p = KvPool{};
        if ((e = hipMalloc(reinterpret_cast<void**>(&p.k), need)) != hipSuccess) {
            p.k = nullptr;
            return {QMM_ERR_HIP, std::string("hipMalloc (KV cache): ") + hipGetErrorString(e)};
        }
        if ((e = hipMalloc(reinterpret_cast<void**>(&p.v), need)) != hipSuccess) {
            (void)hipFree(p.k);
            p = KvPool{};
            return {QMM_ERR_HIP, std::string("hipMalloc (KV cache): ") + hipGetErrorString(e)};
        }
        p.cap = need;
    }
    p.layers = layers;
    p.max_seq = max_seq;
    p.kv_heads = kv_heads;
    p.head_dim = head_dim;
    return {QMM_OK, ""};
}

LayerStatus kv_cache_free() {
    std::lock_guard<std::mutex> lock(g_kv_mutex);
    int cur = 0;
    hipError_t e = hipGetDevice(&cur);
    if (e != hipSuccess) return {QMM_ERR_HIP, std::string("hipGetDevice: ") + hipGetErrorString(e)};
    for (auto& kv : g_kv) {
        if (!kv.second.k) continue;
        if ((e = hipSetDevice(kv.first)) != hipSuccess) return {QMM_ERR_HIP, hipGetErrorString(e)};
        (void)hipDeviceSynchronize();  // queued kernels may still use the pool
        (void)hipFree(kv.second.k);
        (void)hipFree(kv.second.v);
    }
    g_kv.clear();
    (void)hipSetDevice(cur);
    return {QMM_OK, ""};
}

// Device K / V of layer `layer` for a call writing [start, start + q_len), checked against the
// pool's geometry (the reference's DeviceKVCachePool checks, attention.hip:316-331).
LayerStatus kv_cache_layer(int layer, int start, int q_len, int kv_heads, int head_dim, _Float16** k, _Float16** v,
                           int* max_seq) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return {QMM_ERR_HIP, std::string("hipGetDevice: ") + hipGetErrorString(e)};
    std::lock_guard<std::mutex> lock(g_kv_mutex);
    auto it = g_kv.find(dev);
    if (it == g_kv.end() || !it->second.k)
        return {QMM_ERR_UNSUPPORTED, "Device KV cache not initialized. Call kv_cache_init first."};
    const KvPool& p = it->second;
    if (layer < 0 || layer >= p.layers) return {QMM_ERR_OUT_OF_RANGE, "layer_idx out of range for DeviceKVCachePool."};
    if (start < 0 || static_cast<int64_t>(start) + q_len > p.max_seq)
        return {QMM_ERR_OUT_OF_RANGE, "start_pos + q_len exceeds max_seq_len in DeviceKVCachePool."};
    if (kv_heads != p.kv_heads || head_dim != p.head_dim)
        return {QMM_ERR_INVALID_ARGUMENT, "num_kv_heads or head_dim mismatch with DeviceKVCachePool."};
    const size_t layer_elems = static_cast<size_t>(p.max_seq) * p.kv_heads * p.head_dim;
    *k = p.k + static_cast<size_t>(layer) * layer_elems;
    *v = p.v + static_cast<size_t>(layer) * layer_elems;
    if (max_seq) *max_seq = p.max_seq;
    return {QMM_OK, ""};
}

// ---- the layer pipeline --------------------------------------------------------------------
LayerStatus forward_layer(const qmm_layer_config& cfg, const qmm_layer_weights& w, const void* x_in, void* x_out,
                          int layer_idx, int seq_len, int pos_offset, hipStream_t stream) {
    const int H = cfg.num_heads, KVH = cfg.num_kv_heads, D = cfg.head_dim;
    const int hid = cfg.hidden_size, inter = cfg.intermediate_size;
    if (seq_len <= 0 || hid <= 0 || inter <= 0 || H <= 0 || KVH <= 0 || D <= 0)
        return {QMM_ERR_INVALID_ARGUMENT, "seq_len and the layer dimensions must be positive."};
    if (H % KVH != 0) return {QMM_ERR_INVALID_ARGUMENT, "num_heads must be divisible by num_kv_heads."};
    if (D > kMaxHeadDim || D % 2 != 0) return {QMM_ERR_INVALID_ARGUMENT, "head_dim must be even and in (0, 256]."};
    if (x_in == nullptr || x_out == nullptr) return {QMM_ERR_INVALID_ARGUMENT, "x_in and x_out must be non-null."};
    const int qd = H * D, kvd = KVH * D;
    _Float16 *kc = nullptr, *vc = nullptr;
    LayerStatus st = kv_cache_layer(layer_idx, pos_offset, seq_len, KVH, D, &kc, &vc, nullptr);
    if (st.code != QMM_OK) return st;
    const int kv_len = pos_offset + seq_len;

    // activation workspace
    const size_t S = static_cast<size_t>(seq_len);
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t at = off;
        off += (bytes + 255) & ~size_t{255};
        return at;
    };
    const size_t o_norm = take(S * hid * 2), o_q = take(S * qd * 2), o_k = take(S * kvd * 2), o_v = take(S * kvd * 2);
    const size_t o_qr = take(S * qd * 2), o_att = take(S * qd * 2), o_proj = take(S * hid * 2), o_h = take(S * hid * 2);
    const size_t o_g = take(S * inter * 2), o_u = take(S * inter * 2), o_act = take(S * inter * 2);
    const size_t o_down = take(S * hid * 2), o_part = take(attn_plan(seq_len, kv_len, H, KVH, D, pos_offset, true, attn_aligned(kc, vc, nullptr), true).bytes);
    void* ws_buf = nullptr;
    std::unique_lock<std::mutex> ws_held;  // until the layer's last launch
    hipError_t e = take_workspace(WorkspaceKind::kLayer, stream, off, ws_held, &ws_buf);
    if (e != hipSuccess) return {QMM_ERR_HIP, std::string("layer workspace: ") + hipGetErrorString(e)};
    char* const ws = static_cast<char*>(ws_buf);
    auto fail = [](hipError_t err, const char* what) {
        return LayerStatus{QMM_ERR_HIP, std::string(what) + ": " + hipGetErrorString(err)};
    };
    auto gemms = [&](const qmm_gemm_desc* d, int n) -> LayerStatus {
        const int rc = qmm_gemm_batch(d, n, stream);
        if (rc != QMM_OK) return {rc, qmm_last_error()};
        return {QMM_OK, ""};
    };
    auto desc = [&](int t, const void* A, const void* W, void* C, int M, int N, int K) {
        qmm_gemm_desc d{};
        d.ggml_type = t;
        d.A = A;
        d.a_dtype = QMM_DTYPE_F16;
        d.W = W;
        d.C = C;
        d.c_dtype = QMM_DTYPE_F16;
        d.M = M;
        d.N = N;
        d.K = K;
        return d;
    };
    const int nw_f32 = w.attn_norm_dtype == QMM_DTYPE_F32 ? 1 : 0, fw_f32 = w.ffn_norm_dtype == QMM_DTYPE_F32 ? 1 : 0;
    // Decode (one row): the norms, SwiGLU and the last residual add are folded into the GEMV
    // launches (their activation staging and output epilogue); a step whose shapes the folded
    // kernels do not take runs the separate kernels instead.
    const bool fold = seq_len == 1;
    // Runs descriptors of `d` with fold `fz` on their common activations, consecutive descriptors
    // of one weight type as one launch, until one is not supported folded; `done` = how many ran.
    auto folded = [&](const qmm_gemm_desc* d, int n, const GemvFuse& fz, int& done) -> LayerStatus {
        done = 0;
        if (!fold) return {QMM_OK, ""};
        for (int i = 0; i < n;) {
            int j = i + 1;
            while (j < n && d[j].ggml_type == d[i].ggml_type) ++j;
            const void* W[3];
            void* C[3];
            int N[3];
            for (int t = i; t < j; ++t) {
                W[t - i] = d[t].W;
                C[t - i] = d[t].C;
                N[t - i] = d[t].N;
            }
            const hipError_t fe = launch_gemv_ex(d[i].ggml_type, d[i].A, QMM_DTYPE_F16, 1, d[i].K, W, C, N, j - i, fz, stream);
            if (fe == hipErrorNotSupported) return {QMM_OK, ""};  // the caller runs the rest unfolded
            if (fe != hipSuccess) return {QMM_ERR_HIP, std::string("folded GEMV: ") + hipGetErrorString(fe)};
            i = j;
            done = j;
        }
        return {QMM_OK, ""};
    };
    int done = 0;

    // 1.-2. pre-attention RMSNorm, q, k, v (one launch per weight type)
    const qmm_gemm_desc qkv[3] = {desc(w.wq_type, ws + o_norm, w.wq, ws + o_q, seq_len, qd, hid),
                                  desc(w.wk_type, ws + o_norm, w.wk, ws + o_k, seq_len, kvd, hid),
                                  desc(w.wv_type, ws + o_norm, w.wv, ws + o_v, seq_len, kvd, hid)};
    {
        GemvFuse fz;
        fz.kind = 1;
        fz.w = w.attn_norm;
        fz.w_f32 = nw_f32;
        fz.eps = cfg.rms_norm_eps;
        qmm_gemm_desc dq[3] = {qkv[0], qkv[1], qkv[2]};
        for (auto& d : dq) d.A = x_in;
        if ((st = folded(dq, 3, fz, done)).code != QMM_OK) return st;
    }
    if (done < 3) {
        if ((e = launch_rmsnorm(x_in, nullptr, w.attn_norm, nw_f32, nullptr, ws + o_norm, seq_len, hid, cfg.rms_norm_eps,
                                stream)) != hipSuccess)
            return fail(e, "rmsnorm");
        if ((st = gemms(qkv + done, 3 - done)).code != QMM_OK) return st;
    }
    // optional q / k / v biases, added to the projections before the rotation
    {
        const void* const bias[3] = {w.bq, w.bk, w.bv};
        const size_t at[3] = {o_q, o_k, o_v};
        const int bn[3] = {qd, kvd, kvd};
        for (int i = 0; i < 3; ++i)
            if (bias[i] != nullptr && (e = launch_bias_add(ws + at[i], bias[i], seq_len, bn[i], stream)) != hipSuccess)
                return fail(e, "q/k/v bias");
    }
    // 3.-4. RoPE on q and k (k and v land in the cache at their positions), attention over the
    // cache; in decode the rotation and the cache write run inside the attention kernel
    const float scale = cfg.scale != 0.0f ? cfg.scale : 1.0f / std::sqrt(static_cast<float>(D));
    e = fold ? launch_attention_decode_rope(ws + o_q, ws + o_k, ws + o_v, kc, vc, ws + o_att, ws + o_part, kv_len, H, KVH, D,
                                            scale, cfg.rope_freq_base, cfg.rope_neox != 0, stream)
             : hipErrorNotSupported;
    if (e == hipErrorNotSupported) {
        const size_t cache_off = static_cast<size_t>(pos_offset) * kvd;
        if ((e = launch_rope(ws + o_q, ws + o_qr, H, ws + o_k, kc + cache_off, ws + o_v, vc + cache_off, KVH, seq_len, D,
                             pos_offset, cfg.rope_freq_base, cfg.rope_neox != 0, stream)) != hipSuccess)
            return fail(e, "rope");
        e = launch_attention(ws + o_qr, kc, vc, ws + o_att, ws + o_part, seq_len, kv_len, H, KVH, D, pos_offset, scale, true,
                             true, stream);
    }
    if (e != hipSuccess) return fail(e, "attention");
    // 5. output projection
    const qmm_gemm_desc o = desc(w.wo_type, ws + o_att, w.wo, ws + o_proj, seq_len, hid, qd);
    if ((st = gemms(&o, 1)).code != QMM_OK) return st;
    if (w.bo != nullptr && (e = launch_bias_add(ws + o_proj, w.bo, seq_len, hid, stream)) != hipSuccess)
        return fail(e, "output bias");
    // 6.-7. residual + pre-FFN RMSNorm, gate, up (one launch per weight type)
    const qmm_gemm_desc gu[2] = {desc(w.wgate_type, ws + o_norm, w.wgate, ws + o_g, seq_len, inter, hid),
                                 desc(w.wup_type, ws + o_norm, w.wup, ws + o_u, seq_len, inter, hid)};
    bool h_ready = false;    // h = half(x_in + o) materialised at ws + o_h
    bool act_ready = false;  // SwiGLU's output already at ws + o_act
    {
        GemvFuse fz;
        fz.kind = 2;
        fz.R = ws + o_proj;
        fz.w = w.ffn_norm;
        fz.w_f32 = fw_f32;
        fz.eps = cfg.rms_norm_eps;
        qmm_gemm_desc dg[2] = {gu[0], gu[1]};
        for (auto& d : dg) d.A = x_in;
        if (w.wgate_type == w.wup_type) {
            // gate row n and up row n in one wave: the launch writes SwiGLU's output directly
            qmm_gemm_desc dp[2] = {dg[0], dg[1]};
            dp[0].C = ws + o_act;
            fz.pair = 1;
            if ((st = folded(dp, 2, fz, done)).code != QMM_OK) return st;
            act_ready = done == 2;
            fz.pair = 0;
        }
        if (!act_ready && (st = folded(dg, 2, fz, done)).code != QMM_OK) return st;
    }
    if (!act_ready && done < 2) {
        if ((e = launch_rmsnorm(x_in, ws + o_proj, w.ffn_norm, fw_f32, ws + o_h, ws + o_norm, seq_len, hid,
                                cfg.rms_norm_eps, stream)) != hipSuccess)
            return fail(e, "rmsnorm_residual");
        h_ready = true;
        if ((st = gemms(gu + done, 2 - done)).code != QMM_OK) return st;
    }
    // 8.-9. SwiGLU (unless the gate/up launch produced it), down and the second residual (folded
    // into down's output).  SwiGLU is not folded into down's staging: every down workgroup would
    // read both intermediate vectors and evaluate every exp (measured slower than a kernel).
    if (!act_ready &&
        (e = launch_swiglu(ws + o_g, ws + o_u, ws + o_act, static_cast<int64_t>(S) * inter, stream)) != hipSuccess)
        return fail(e, "swiglu");
    {
        GemvFuse fz;
        fz.ea = x_in;
        fz.eb = ws + o_proj;
        const qmm_gemm_desc dd = desc(w.wdown_type, ws + o_act, w.wdown, x_out, seq_len, hid, inter);
        if ((st = folded(&dd, 1, fz, done)).code != QMM_OK) return st;
    }
    if (done < 1) {
        const qmm_gemm_desc dn = desc(w.wdown_type, ws + o_act, w.wdown, ws + o_down, seq_len, hid, inter);
        if ((st = gemms(&dn, 1)).code != QMM_OK) return st;
        if (!h_ready &&
            (e = launch_residual_add(x_in, ws + o_proj, ws + o_h, static_cast<int64_t>(S) * hid, stream)) != hipSuccess)
            return fail(e, "residual_add");
        if ((e = launch_residual_add(ws + o_h, ws + o_down, x_out, static_cast<int64_t>(S) * hid, stream)) != hipSuccess)
            return fail(e, "residual_add");
    }
    return {QMM_OK, ""};
}

}  // namespace qmm
