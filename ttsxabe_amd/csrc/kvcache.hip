// KV-cache producers: RoPE, append (f32 / f16 / Q8_0), fused rotate+append,
// and growth, all writing the layouts the attention kernels read.
//
// Replaces crates/llmtie-cuda/src/kernels.rs:4908-4948 (`rope`),
// :5244-5318 (`cache_append[_t][_f16]`), :5334-5380 (`rope_cache_f16`) and
// :5397-5423 (`cache_grow[_f16]`). The Q8_0 producers have no reference
// counterpart (the reference holds no quantized KV cache); they quantize as
// ggml's `quantize_row_q8_0_ref` does: d = max|x| / 127, code = round-half-
// away(x / d), d stored as f16, one block per 32 dims of one position.
//
// One token's producers are launch-bound: a flat index per element, coalesced
// over the source row, scattered into the destination layout. Over the rows of
// a prompt they are bound by memory, and the kernels for that say how.
#include <algorithm>

#include "common.h"
#include "kvcache.h"
#include "kvlayout.h"

// No multiply-add contraction in this file: the rotations are the reference's
// separate f32 multiplies and subtraction, so the fused rotate+append and the
// separate rope then append produce the same bits whatever the kernel.
#pragma clang fp contract(off)

namespace llmtie {

constexpr int KB = 256;

// RoPE angle of pair j at position p, in f32 as the reference's CPU twin
// (crates/llmtie-dsp/src/rope.rs:83-126) computes it.
__device__ __forceinline__ void rope_sc(int j, int hd, float theta, const float* div, int p, float& sn, float& cs) {
    float inv = powf(theta, -2.0f * (float)j / (float)hd);
    if (div) inv /= div[j];
    sincosf((float)p * inv, &sn, &cs);
}

// RoPE in place over x[off ..] of [t, heads * hd], halves paired. What bounded
// the flat form (a pair a thread) was not its bytes but its powf and sincosf,
// which every head of a position repeated. Here a workgroup takes pn positions
// by jn pairs (pn * jn <= KB), each thread evaluates one angle into LDS, and
// the workgroup then streams `hpb` heads of those positions: thread
// (hl, p, jv) keeps the VEC angles of its pairs in registers and walks the
// heads hl, hl + HL, .. with VEC-wide loads of both halves, UN heads in
// flight; the first loads go out before the angles are evaluated. The values
// are the flat form's bit for bit (the same two products and sum of the same
// sine and cosine). VEC = 4 wants half a head in whole aligned float4s; VEC = 1
// takes any even head and any alignment.
// Kernel times, flat form -> this: 8192 rows of 32 heads of 128, 120 -> 45 us
// (6.0 TB/s of reads and writes, what a large copy reaches); of 8 heads, 31 ->
// 12.7; 1999 rows of 32 heads, 33 -> 11.9; 3001 rows of 8 heads, 16.0 -> 8.3.
template <int VEC, int HD>
__global__ __launch_bounds__(KB) void rope_kernel(float* x, long off, const float* div, int t, int heads, int hd_,
                                                  float theta, int first, int pn_, int jn_, int tiles, int groups,
                                                  int hpb) {
    constexpr int UN = VEC == 4 ? 2 : 4;  // heads in flight
    __shared__ float2 ang[KB];
    // HD > 0: the head width is known, one pair chunk, and the position tile
    // and head group are the grid's; 0: any width, one index over all three.
    const int hd = HD ? HD : hd_, half = hd >> 1;
    const int jn = HD ? half : jn_, pn = HD ? KB / jn : pn_;
    int tile = (int)blockIdx.x, grp = (int)blockIdx.y, j0 = 0;
    if constexpr (HD == 0) {
        tile = (int)(blockIdx.x % (unsigned)tiles);
        grp = (int)(blockIdx.x / (unsigned)tiles % (unsigned)groups);
        j0 = (int)(blockIdx.x / (unsigned)tiles / (unsigned)groups) * jn;
    }
    const int jv = jn / VEC;    // vectors of one position
    const int span = pn * jv;   // threads of one head
    const int hl = (int)threadIdx.x / span, e = (int)threadIdx.x % span;
    const int nhl = KB / span;  // heads side by side
    const int pl = e / jv, jl = e % jv * VEC;
    const int p = tile * pn + pl;
    const int h1 = min(heads, (grp + 1) * hpb);
    const bool live = hl < nhl && p < t && j0 + jl < half;
    float* row = x + (size_t)off + (size_t)(live ? p : 0) * heads * hd + (live ? j0 + jl : 0);
    typedef float vec __attribute__((ext_vector_type(VEC)));
    int h = live ? grp * hpb + hl : h1;
    vec a[UN], b[UN];
    auto load = [&](int h0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            if (h0 + u * nhl < h1) {
                const float* r = row + (size_t)(h0 + u * nhl) * hd;
                a[u] = *reinterpret_cast<const vec*>(r);
                b[u] = *reinterpret_cast<const vec*>(r + half);
            }
        }
    };
    load(h);
    if ((int)threadIdx.x < pn * jn) {
        float2 sc;
        // Pairs past the half (a ragged last chunk) repeat its last one.
        rope_sc(min(j0 + (int)threadIdx.x % jn, half - 1), hd, theta, div,
                first + tile * pn + (int)threadIdx.x / jn, sc.x, sc.y);
        ang[threadIdx.x] = sc;
    }
    __syncthreads();
    vec sn, cs;
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
        const float2 sc = ang[live ? pl * jn + jl + i : 0];
        sn[i] = sc.x;
        cs[i] = sc.y;
    }
    while (h < h1) {
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            if (h + u * nhl < h1) {
                float* r = row + (size_t)(h + u * nhl) * hd;
                *reinterpret_cast<vec*>(r) = a[u] * cs - b[u] * sn;
                *reinterpret_cast<vec*>(r + half) = b[u] * cs + a[u] * sn;
            }
        }
        h += UN * nhl;
        load(h);
    }
}

// f32 or f16 append of n rows [n][kv*hd] into K [kv][cap][hd] or (transposed)
// V [kv][hd][cap] at positions past..past+n-1.
template <typename T, bool TR>
__global__ __launch_bounds__(KB) void append_kernel(const float* src, T* dst, int n, int kv, int hd,
                                                    int cap, int past) {
    const long i = (long)blockIdx.x * KB + threadIdx.x;
    const int d = kv * hd;
    if (i >= (long)n * d) return;
    const int ti = (int)(i / d);
    const int hh = (int)((i % d) / hd);
    const int j = (int)(i % hd);
    const float x = src[i];
    const size_t at = TR ? ((size_t)hh * hd + j) * cap + past + ti : ((size_t)hh * cap + past + ti) * hd + j;
    if constexpr (sizeof(T) == 2) {
        dst[at] = __builtin_bit_cast(uint16_t, to_h(x));
    } else {
        dst[at] = x;
    }
}

// append_kernel's K orientation eight dims a thread: two float4 in, one (f16)
// or two (f32) 16-byte stores out, where head rows and both buffers are
// aligned for it. 1999 rows of 8 heads of 128 into f16: 6.4 -> 4.4 us.
template <typename T>
__global__ __launch_bounds__(KB) void append_k8_kernel(const float* src, T* dst, unsigned total8, unsigned d8,
                                                       unsigned hd8, int cap, int past) {
    const unsigned i = blockIdx.x * (unsigned)KB + threadIdx.x;
    if (i >= total8) return;
    const unsigned ti = i / d8, c = i - ti * d8;
    const unsigned hh = c / hd8, j = c - hh * hd8;
    const float4* in = reinterpret_cast<const float4*>(src) + (size_t)i * 2;
    const float4 lo = in[0], hi = in[1];
    T* at = dst + (((size_t)hh * cap + past + ti) * hd8 + j) * 8;
    if constexpr (sizeof(T) == 2) {
        half8 h;
        h[0] = to_h(lo.x), h[1] = to_h(lo.y), h[2] = to_h(lo.z), h[3] = to_h(lo.w);
        h[4] = to_h(hi.x), h[5] = to_h(hi.y), h[6] = to_h(hi.z), h[7] = to_h(hi.w);
        *reinterpret_cast<half8*>(at) = h;
    } else {
        reinterpret_cast<float4*>(at)[0] = lo;
        reinterpret_cast<float4*>(at)[1] = hi;
    }
}

// append_kernel's V orientation over many rows: the flat form's neighbouring
// threads hold neighbouring dims, so each store of a wave touched 64 cache
// rows. A workgroup takes a tile of AT_P positions by AT_D dims through LDS:
// rows read as float4s, then four positions of one dim a thread, stored
// together where `wide` (cap and base aligned) says so. Tiles lie on multiples
// of AT_P positions, so a tile's stores fill whole 128-byte (f16) runs of a
// cache row; positions outside past .. past + n - 1 are left as they are.
// 1999 rows of 8 heads of 128 into f16: 13.6 -> 3.9 us; 173 rows: 4.6 either way (latency).
constexpr int AT_P = 64, AT_D = 32;
template <typename T>
__global__ __launch_bounds__(KB) void append_vt_kernel(const float* src, T* dst, int n, int d, int cap, int past,
                                                       int wide) {
    __shared__ float tile[AT_D][AT_P + 1];
    const int d0 = blockIdx.y * AT_D;
    const int p0 = (past / AT_P + (int)blockIdx.x) * AT_P;  // the tile's first position
#pragma unroll
    for (int r = 0; r < AT_P * AT_D / 4 / KB; ++r) {
        const int e = (int)threadIdx.x + r * KB;
        const int q = e % (AT_D / 4), pl = e / (AT_D / 4);
        const int ti = pl + (p0 - past);  // p0 + pl may pass an int
        if (ti < 0 || ti >= n) continue;
        const float4 x = *reinterpret_cast<const float4*>(src + (size_t)ti * d + d0 + 4 * q);
        tile[4 * q][pl] = x.x;
        tile[4 * q + 1][pl] = x.y;
        tile[4 * q + 2][pl] = x.z;
        tile[4 * q + 3][pl] = x.w;
    }
    __syncthreads();
    typedef T quad __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int r = 0; r < AT_P * AT_D / 4 / KB; ++r) {
        const int e = (int)threadIdx.x + r * KB;
        const int pl = e % (AT_P / 4) * 4, dl = e / (AT_P / 4);
        const int ti = pl + (p0 - past);
        T* at = dst + (size_t)(d0 + dl) * cap + p0 + pl;
        quad y;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float x = tile[dl][pl + i];
            if constexpr (sizeof(T) == 2) y[i] = __builtin_bit_cast(uint16_t, to_h(x));
            else y[i] = x;
        }
        if (wide && ti >= 0 && ti + 4 <= n) {
            *reinterpret_cast<quad*>(at) = y;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (ti + i >= 0 && ti + i < n) at[i] = y[i];
        }
    }
}

// The one-token kernels below (rotate and store) are a launch, a memory round
// trip and an angle: with the head width known (HD; 0: any) the index
// arithmetic is shifts, and the row's values are loaded before the angle is
// evaluated, so the two overlap. 32/8/128 in a graph of launches (a fill of the
// same size takes 1.85 us): f16 2.46 -> 2.30 us, tiled 2.47 -> 2.34, Q8_0 (its
// block maxima on DPP, not LDS shuffles) 2.77 -> 2.56.
//
// The pair of element e of a row of heads, rotated at position p.
__device__ __forceinline__ float2 rotated_pair(const float* row, int hh, int j, int hd, float theta, const float* div,
                                               int p) {
    const int half = hd >> 1;
    const float a0 = row[(size_t)hh * hd + j], b0 = row[(size_t)hh * hd + j + half];
    __builtin_amdgcn_sched_barrier(0);
    float sn, cs;
    rope_sc(j, hd, theta, div, p, sn, cs);
    return make_float2(a0 * cs - b0 * sn, b0 * cs + a0 * sn);
}

// q rotated in place; k rotated and v copied into the f16 caches at `pos`.
template <int HD>
__global__ __launch_bounds__(KB) void rope_cache_f16_kernel(float* q, const float* k, const float* v, const float* div,
                                                            int heads, int kv, int hd_, float theta, int pos,
                                                            uint16_t* kc, uint16_t* vc, int cap) {
    const int hd = HD ? HD : hd_, half = hd >> 1;
    const int nq = heads * half, nk = kv * half, nv = kv * hd;
    const int i = blockIdx.x * KB + threadIdx.x;
    if (i < nq + nk) {
        const bool is_q = i < nq;
        const int e = is_q ? i : i - nq;
        const int j = e % half, hh = e / half;
        const float2 y = rotated_pair(is_q ? q : k, hh, j, hd, theta, div, pos);
        if (is_q) {
            float* d = q + (size_t)hh * hd + j;
            d[0] = y.x;
            d[half] = y.y;
        } else {
            uint16_t* d = kc + ((size_t)hh * cap + pos) * hd + j;
            d[0] = __builtin_bit_cast(uint16_t, to_h(y.x));
            d[half] = __builtin_bit_cast(uint16_t, to_h(y.y));
        }
    } else if (i < nq + nk + nv) {
        const int e = i - nq - nk;
        vc[(size_t)e * cap + pos] = __builtin_bit_cast(uint16_t, to_h(v[e]));
    }
}

template <typename T>
__global__ __launch_bounds__(KB) void grow_kernel(const T* src, T* dst, int rows, int len, int ss, int ds) {
    const long i = (long)blockIdx.x * KB + threadIdx.x;
    if (i >= (long)rows * len) return;
    const int r = (int)(i / len), j = (int)(i % len);
    dst[(size_t)r * ds + j] = src[(size_t)r * ss + j];
}

// Row-wide (16 lanes) maximum, every lane getting it: DPP within the row.
__device__ __forceinline__ float row_max(float v) {
    v = fmaxf(v, dpp_f<0xb1>(v));   // quad_perm [1,0,3,2]
    v = fmaxf(v, dpp_f<0x4e>(v));   // quad_perm [2,3,0,1]
    v = fmaxf(v, dpp_f<0x141>(v));  // row_half_mirror
    return fmaxf(v, dpp_f<0x140>(v));  // row_mirror
}

// One Q8_0 block per 32 consecutive threads: the 32 dims [32b, 32b+32) of
// one (position, kv head) row. `x` is this thread's element.
__device__ __forceinline__ void q8_block(float x, int8_t& code, uint16_t& dbits) {
    // Every lane of the wave takes part (DPP reads them all).
    const float r = row_max(fabsf(x));
    const auto w = __builtin_amdgcn_permlane16_swap(__float_as_uint(r), __float_as_uint(r), false, false);
    const float amax = fmaxf(__uint_as_float(w[0]), __uint_as_float(w[1]));
    const float d = amax / 127.0f;
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    code = (int8_t)(int)roundf(x * id);
    dbits = __builtin_bit_cast(uint16_t, to_h(d));
}

// Byte offsets of element (position p, dim d) of (slot, kv head) `kvh` in a
// tiled Q8_0 cache (kvlayout.h): codes and the scale of its dim block.
struct Q8At {
    long code, scale;
};
__device__ __forceinline__ Q8At q8_at(size_t kvh, int nblk, int hd, int p, int d, bool value) {
    const long blk = ((long)kvh * nblk + (p >> 5)) * tq8_block_bytes(hd);
    const int kk = p & 31;
    Q8At r;
    r.code = blk + (value ? 32L * hd + tq8_v_off(kk, d) : tq8_k_off(hd, kk, d));
    r.scale = blk + 64L * hd + (value ? 64L * (hd / 32) : 0) + 2L * ((d >> 5) * 32 + kk);
    return r;
}

// n rows [n][kv*hd] of K (already rotated) and V into slot `slot` of a tiled
// Q8_0 cache at positions past..past+n-1.
__global__ __launch_bounds__(KB) void append_q8_kernel(const float* k, long k_off, const float* v, long v_off,
                                                       char* cache, int slot, int n, int kv, int hd, int cap,
                                                       int past) {
    const long i = (long)blockIdx.x * KB + threadIdx.x;
    const int d = kv * hd;
    const long total = (long)n * d;
    // Threads past the end still take part in the block-wide shuffles as
    // zeros; total is a multiple of 32, so they are whole groups.
    const bool live = i < total;
    const long ii = live ? i : 0;
    const int ti = (int)(ii / d);
    const int hh = (int)((ii % d) / hd);
    const int j = (int)(ii % hd);
    const size_t kvh = (size_t)slot * kv + hh;
    const int nb = tiled_nblk(cap);
    int8_t c;
    uint16_t db;
    q8_block(live ? k[k_off + ii] : 0.0f, c, db);
    if (live) {
        const Q8At at = q8_at(kvh, nb, hd, past + ti, j, false);
        cache[at.code] = (char)(c ^ 0x80);
        if ((j & 31) == 0) *reinterpret_cast<uint16_t*>(cache + at.scale) = db;
    }
    q8_block(live ? v[v_off + ii] : 0.0f, c, db);
    if (live) {
        const Q8At at = q8_at(kvh, nb, hd, past + ti, j, true);
        cache[at.code] = (char)(c ^ 0x80);
        if ((j & 31) == 0) *reinterpret_cast<uint16_t*>(cache + at.scale) = db;
    }
}

// d and 1 / d of a block's largest magnitude, as q8_block takes them.
__device__ __forceinline__ float q8_scale(float amax, float& id) {
    const float d = amax / 127.0f;
    id = d != 0.0f ? 1.0f / d : 0.0f;
    return d;
}

// A code as the cache stores it: offset binary.
__device__ __forceinline__ uint32_t q8_code(float x, float id) {
    return (uint32_t)(uint8_t)(int8_t)(int)roundf(x * id) ^ 0x80u;
}

// The positions of past .. past + n - 1 whose eight-position V chunk is not
// wholly appended: `lead` from past on, then `trail` up to the end. The chunk
// kernels leave them to workgroups of their own that store element by element
// as the flat forms do (predicated stores of a chunk's 32 values in one lane
// held a launch of few rows up by 0.7 us).
struct Edges {
    int lead, trail;
    __host__ __device__ Edges(int past, int n) {
        const int end = past + n, up = (past + 7) / 8 * 8, down = end / 8 * 8;
        lead = (up < end ? up : end) - past;
        trail = down >= up ? end - down : 0;
    }
    __host__ __device__ int count() const { return lead + trail; }
    // Row (of the appended ones) of edge position e.
    __device__ int row(int e, int n) const { return e < lead ? e : n - trail + (e - lead); }
};

// append_q8_kernel in whole fragment chunks, for sources aligned to 16 bytes
// (the cache's blocks are): the flat form stored one byte a thread and reduced
// each block of 32 through LDS shuffles. One wave takes, of one block of one
// kv head, either a K unit (key tile T, 64 dims: lane (key m, group g) holds 8
// + 8 dims of one key, whose blocks of 32 are the four lanes of its column) or
// a V unit (32 dims: lane (dim col, group g) holds dims col and col + 16 of
// eight keys, whose blocks are the 16 lanes of its row). Every lane stores 16
// bytes of codes, 1 KB contiguous a wave; V chunks cut by past or past + n
// store their own positions one by one. The codes and scales are the flat
// form's: a maximum does not depend on its order.
// 3001 rows of 8 heads of 128 (25 MB read, 6.5 written): 22.6 -> 9.0 us.
__global__ __launch_bounds__(KB) void append_q8_chunks_kernel(const float* k, const float* v, char* cache, int slot,
                                                              int n, int kv, int hd, int nblk, int past, int units,
                                                              int b0) {
    const int ns = hd / 32;  // K units of a block, and V units
    const size_t d = (size_t)kv * hd;
    const int uwgs = (units + KB / 64 - 1) / (KB / 64);
    if ((int)blockIdx.x >= uwgs) {
        const Edges ed(past, n);
        const long i = (long)((int)blockIdx.x - uwgs) * KB + threadIdx.x;
        const bool live = i < (long)(ed.count() * d);  // whole groups of 32 threads
        const int ti = live ? ed.row((int)(i / (long)d), n) : 0, c = live ? (int)(i % (long)d) : 0;
        int8_t code;
        uint16_t db;
        q8_block(live ? v[ti * d + c] : 0.0f, code, db);
        if (!live) return;
        const Q8At at = q8_at((size_t)slot * kv + c / hd, nblk, hd, past + ti, c % hd, true);
        cache[at.code] = (char)(code ^ 0x80);
        if ((c & 31) == 0) *reinterpret_cast<uint16_t*>(cache + at.scale) = db;
        return;
    }
    const int w = (int)blockIdx.x * (KB / 64) + (int)(threadIdx.x >> 6);
    if (w >= units) return;
    const int l = threadIdx.x & 63, col = l & 15, g = l >> 4;
    const int u = w % (2 * ns), hh = w / (2 * ns) % kv, b = w / (2 * ns) / kv + b0;
    char* blk = cache + (((size_t)slot * kv + hh) * nblk + b) * tq8_block_bytes(hd);
    if (u < ns) {
        const int T = u / (ns / 2), sp = u % (ns / 2);
        const int kk = 8 * (col >> 2) + 4 * T + (col & 3), ti = b * 32 + kk - past;
        const bool live = ti >= 0 && ti < n;
        // The four lanes of a column share a key, so they are live together.
        const float4* in = reinterpret_cast<const float4*>(k + (live ? ti : 0) * d + (size_t)hh * hd + 64 * sp + 8 * g);
        const float4 x[4] = {in[0], in[1], in[8], in[9]};
        uint32_t code[4];
        uint16_t dh[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const float4 a = x[2 * s], c = x[2 * s + 1];
            const float m = fmaxf(fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))),
                                  fmaxf(fmaxf(fabsf(c.x), fabsf(c.y)), fmaxf(fabsf(c.z), fabsf(c.w))));
            float id;
            dh[s] = __builtin_bit_cast(uint16_t, to_h(q8_scale(max4grp(m), id)));
            code[2 * s] = q8_code(a.x, id) | q8_code(a.y, id) << 8 | q8_code(a.z, id) << 16 | q8_code(a.w, id) << 24;
            code[2 * s + 1] = q8_code(c.x, id) | q8_code(c.y, id) << 8 | q8_code(c.z, id) << 16 | q8_code(c.w, id) << 24;
        }
        if (!live) return;
        *reinterpret_cast<uint4*>(blk + ((size_t)u * 64 + l) * 16) = make_uint4(code[0], code[1], code[2], code[3]);
        if (g < 2) reinterpret_cast<uint16_t*>(blk + 64 * hd)[(2 * sp + g) * 32 + kk] = g ? dh[1] : dh[0];
    } else {
        const int tp = u - ns;  // dims 32 tp ..
        const int t0 = b * 32 + 8 * g - past;
        float x0[8], x1[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            // A lane of a cut chunk repeats appended rows and stores nothing
            // (the row maxima run over whole rows of lanes, one chunk each).
            const float* in = v + min(max(t0 + j, 0), n - 1) * d + (size_t)hh * hd + 32 * tp + col;
            x0[j] = in[0];
            x1[j] = in[16];
        }
        uint32_t code[4] = {0, 0, 0, 0};
        uint16_t dh[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            float id;
            dh[j] = __builtin_bit_cast(uint16_t, to_h(q8_scale(row_max(fmaxf(fabsf(x0[j]), fabsf(x1[j]))), id)));
            code[j >> 2] |= q8_code(x0[j], id) << (8 * (j & 3));
            code[2 + (j >> 2)] |= q8_code(x1[j], id) << (8 * (j & 3));
        }
        char* at = blk + 32 * hd + ((size_t)tp * 64 + l) * 16;
        uint16_t* sc = reinterpret_cast<uint16_t*>(blk + 64 * hd + 2 * hd) + tp * 32 + 8 * g;
        if (t0 < 0 || t0 + 8 > n) return;
        *reinterpret_cast<uint4*>(at) = make_uint4(code[0], code[1], code[2], code[3]);
        if (col == 0) {
            *reinterpret_cast<uint4*>(sc) = make_uint4(dh[0] | (uint32_t)dh[1] << 16, dh[2] | (uint32_t)dh[3] << 16,
                                                       dh[4] | (uint32_t)dh[5] << 16, dh[6] | (uint32_t)dh[7] << 16);
        }
    }
}

// The Q8_0 twin of rope_cache_f16: q rotated in place, k rotated and
// quantized, v quantized, into slot `slot` at position `pos`. Thread e owns
// output element e of the rotated k row (or, past nk, of v), so a block of
// 32 consecutive threads is one Q8_0 block.
template <int HD>
__global__ __launch_bounds__(KB) void rope_cache_q8_kernel(float* q, const float* k, const float* v, const float* div,
                                                           int heads, int kv, int hd_, float theta, int pos,
                                                           char* cache, int slot, int cap) {
    const int hd = HD ? HD : hd_, half = hd >> 1;
    const int nq = heads * half;  // q pairs
    const int nk = kv * hd;       // rotated k elements
    const int nv = kv * hd;
    // Blocks [0, qb) rotate q; the rest quantize k then v. Keeping the two
    // phases in different blocks keeps each k/v block of 32 threads whole.
    const int qblocks = (nq + KB - 1) / KB;
    if ((int)blockIdx.x < qblocks) {
        const int i = blockIdx.x * KB + threadIdx.x;
        if (i >= nq) return;
        const int j = i % half, hh = i / half;
        const float2 y = rotated_pair(q, hh, j, hd, theta, div, pos);
        float* d = q + (size_t)hh * hd + j;
        d[0] = y.x;
        d[half] = y.y;
        return;
    }
    const int i = (blockIdx.x - qblocks) * KB + threadIdx.x;
    const bool live = i < nk + nv;
    const bool is_k = i < nk;
    const int e = live ? (is_k ? i : i - nk) : 0;
    const int hh = e / hd, jj = e % hd;
    float x = 0.0f;
    if (live && is_k) {
        const float2 y = rotated_pair(k, hh, jj % half, hd, theta, div, pos);
        x = jj < half ? y.x : y.y;
    } else if (live) {
        x = v[e];
    }
    int8_t c;
    uint16_t db;
    q8_block(x, c, db);
    if (!live) return;
    const Q8At at = q8_at((size_t)slot * kv + hh, tiled_nblk(cap), hd, pos, jj, !is_k);
    cache[at.code] = (char)(c ^ 0x80);
    if ((jj & 31) == 0) *reinterpret_cast<uint16_t*>(cache + at.scale) = db;
}

// ------------------------------------------------------------ tiled f16

// Half offset of element (position p, dim d) of kv head h in a tiled f16 cache.
__device__ __forceinline__ long t16_at(int h, int nblk, int hd, int p, int d, bool value) {
    const long blk = ((long)h * nblk + (p >> 5)) * 64L * hd;
    return blk + (value ? 32L * hd + t16_v_off(p & 31, d) : t16_k_off(hd, p & 31, d));
}

// The tiled twin of cache_append_f16: n rows [n][kv*hd] into positions
// past.. of the K (or, `value`, the V) area.
__global__ __launch_bounds__(KB) void append_t16_kernel(const float* src, long src_off, uint16_t* cache, int n,
                                                        int kv, int hd, int cap, int past, int value) {
    const long i = (long)blockIdx.x * KB + threadIdx.x;
    const int d = kv * hd;
    if (i >= (long)n * d) return;
    const int ti = (int)(i / d);
    const int hh = (int)((i % d) / hd);
    const int j = (int)(i % hd);
    cache[t16_at(hh, tiled_nblk(cap), hd, past + ti, j, value)] =
        __builtin_bit_cast(uint16_t, to_h(src[src_off + i]));
}

// append_t16_kernel in whole fragment chunks, for sources aligned to 16 bytes
// (the cache's blocks are). One wave takes a 32-position block's K chunk rows
// or V dims of one kv head, each lane 16-byte stores:
//   K: the wave's unit is (key tile T, 32 dims s), lane (key m, group g) eight
//      dims of one key: two float4 in, one chunk out, 1 KB contiguous a wave.
//   V: the unit is 64 dims, lane (dim quad, group g) four dims of eight keys:
//      eight float4 in (256 contiguous bytes of four rows an instruction),
//      four chunks out. Chunks cut by past or past + n are left to the
//      workgroups past the units' (Edges).
// hd / 16 units a block for K, hd / 64 for V.
// 8192 rows of 8 heads of 128 (33 MB read, 17 written): K 26 -> 9.3 us, V
// 31 -> 13.9 us.
template <bool VALUE>
__global__ __launch_bounds__(KB) void append_t16_chunks_kernel(const float* src, uint16_t* cache, int n, int kv,
                                                               int hd, int nblk, int past, int units, int b0) {
    const int per = VALUE ? hd / 64 : hd / 16;  // units of one block
    const int d = kv * hd;
    const int uwgs = (units + KB / 64 - 1) / (KB / 64);
    if (VALUE && (int)blockIdx.x >= uwgs) {
        const Edges ed(past, n);
        const long i = (long)((int)blockIdx.x - uwgs) * KB + threadIdx.x;
        if (i >= (long)ed.count() * d) return;
        const int ti = ed.row((int)(i / d), n), c = (int)(i % d);
        cache[t16_at(c / hd, nblk, hd, past + ti, c % hd, true)] =
            __builtin_bit_cast(uint16_t, to_h(src[(size_t)ti * d + c]));
        return;
    }
    const int w = (int)blockIdx.x * (KB / 64) + (int)(threadIdx.x >> 6);
    if (w >= units) return;
    const int l = threadIdx.x & 63;
    const int u = w % per, hh = w / per % kv, b = w / per / kv + b0;
    uint16_t* blk = cache + ((size_t)hh * nblk + b) * 64 * hd;
    const float* rows = src + (size_t)hh * hd;
    if constexpr (!VALUE) {
        const int ns = hd / 32, T = u / ns, s = u % ns;
        const int m = l & 15, g = l >> 4;
        const int ti = b * 32 + 8 * (m >> 2) + 4 * T + (m & 3) - past;
        if (ti < 0 || ti >= n) return;
        const float4* in = reinterpret_cast<const float4*>(rows + (size_t)ti * d + 32 * s + 8 * g);
        const float4 lo = in[0], hi = in[1];
        half8 h;
        h[0] = to_h(lo.x), h[1] = to_h(lo.y), h[2] = to_h(lo.z), h[3] = to_h(lo.w);
        h[4] = to_h(hi.x), h[5] = to_h(hi.y), h[6] = to_h(hi.z), h[7] = to_h(hi.w);
        *reinterpret_cast<half8*>(blk + ((size_t)u * 64 + l) * 8) = h;
    } else {
        const int q = l & 15, g = l >> 4;  // dims 64u + 4q .., keys 8g ..
        const int t0 = b * 32 + 8 * g - past;
        if (t0 < 0 || t0 + 8 > n) return;
        float4 x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            x[j] = *reinterpret_cast<const float4*>(rows + (size_t)(t0 + j) * d + 64 * u + 4 * q);
        __builtin_amdgcn_sched_barrier(0);  // all eight rows in flight
        const int t = 4 * u + (q >> 2), c = 4 * (q & 3);
        uint16_t* at = blk + 32 * hd + ((size_t)t * 64 + c + 16 * g) * 8;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            half8 h;
#pragma unroll
            for (int j = 0; j < 8; ++j) h[j] = to_h(i == 0 ? x[j].x : i == 1 ? x[j].y : i == 2 ? x[j].z : x[j].w);
            *reinterpret_cast<half8*>(at + 8 * i) = h;
        }
    }
}

// The tiled twin of rope_cache_f16.
template <int HD>
__global__ __launch_bounds__(KB) void rope_cache_t16_kernel(float* q, const float* k, const float* v, const float* div,
                                                            int heads, int kv, int hd_, float theta, int pos,
                                                            uint16_t* cache, int cap) {
    const int hd = HD ? HD : hd_, half = hd >> 1;
    const int nq = heads * half, nk = kv * half, nv = kv * hd;
    const int nb = tiled_nblk(cap);
    const int i = blockIdx.x * KB + threadIdx.x;
    if (i < nq + nk) {
        const bool is_q = i < nq;
        const int e = is_q ? i : i - nq;
        const int j = e % half, hh = e / half;
        const float2 y = rotated_pair(is_q ? q : k, hh, j, hd, theta, div, pos);
        if (is_q) {
            float* d = q + (size_t)hh * hd + j;
            d[0] = y.x;
            d[half] = y.y;
        } else {
            cache[t16_at(hh, nb, hd, pos, j, false)] = __builtin_bit_cast(uint16_t, to_h(y.x));
            cache[t16_at(hh, nb, hd, pos, j + half, false)] = __builtin_bit_cast(uint16_t, to_h(y.y));
        }
    } else if (i < nq + nk + nv) {
        const int e = i - nq - nk;
        cache[t16_at(e / hd, nb, hd, pos, e % hd, true)] = __builtin_bit_cast(uint16_t, to_h(v[e]));
    }
}

// Reference-layout f16 caches (K [kv][cap][hd], V [kv][hd][cap]) into the
// tiled layout, positions 0..live-1 (the rest of the last block is zeroed).
__global__ __launch_bounds__(KB) void ref_to_t16_kernel(const uint16_t* k, const uint16_t* v, uint16_t* cache, int kv,
                                                        int hd, int cap, int live, int tcap) {
    const long i = (long)blockIdx.x * KB + threadIdx.x;
    const int nbl = (live + 31) / 32;
    const long per = (long)nbl * 32 * hd;  // elements per head and area
    if (i >= 2L * kv * per) return;
    const bool value = i >= (long)kv * per;
    const long e = value ? i - (long)kv * per : i;
    const int hh = (int)(e / per);
    const int p = (int)((e % per) / hd), d = (int)(e % hd);
    uint16_t x = 0;
    if (p < live) x = value ? v[((size_t)hh * hd + d) * cap + p] : k[((size_t)hh * cap + p) * hd + d];
    cache[t16_at(hh, tiled_nblk(tcap), hd, p, d, value)] = x;
}

static inline unsigned nblk(long n) { return (unsigned)((n + KB - 1) / KB); }
// Workgroups of an append in whole chunks: a wave a unit, then the edges'
// elements. Past CHUNK_WGS a launch would reach 2^32 threads (two to seven rows
// over two blocks of half a billion dims), where the flat form still has room.
static inline long chunk_wgs(long units, long edges) { return (units + KB / 64 - 1) / (KB / 64) + (edges + KB - 1) / KB; }
constexpr long CHUNK_WGS = (1L << 32) / KB - 1;
static inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

hipError_t launch_rope(float* x, long off, const float* div, int t, int heads, int hd, float theta, int first,
                       hipStream_t st) {
    const int half = hd / 2;
    if ((long)t * heads * half == 0) return hipSuccess;
    // The kernel counts in ints and a launch holds fewer than 2^32 threads:
    // rows of more than 2^23 workgroups, or heads past 2^30, go in halves.
    const bool many = heads > 1 << 30;
    if (t > 1 && (many || (long)t * ((half + KB - 1) / KB) > 1L << 23)) {
        const int lo = t / 2;
        if (hipError_t e = launch_rope(x, off, div, lo, heads, hd, theta, first, st)) return e;
        return launch_rope(x, off + (long)lo * heads * hd, div, t - lo, heads, hd, theta, first + lo, st);
    }
    if (many) {
        const int lo = heads / 2;
        if (hipError_t e = launch_rope(x, off, div, t, lo, hd, theta, first, st)) return e;
        return launch_rope(x, off + (long)lo * hd, div, t, heads - lo, hd, theta, first, st);
    }
    // float4 halves where every head's two halves start on one.
    const int vec = half % 4 == 0 && aligned16(x + off) ? 4 : 1;
    // One angle a thread: jn pairs (whole vectors) of pn positions.
    const int jn = half < KB ? half : KB, chunks = (half + jn - 1) / jn;
    const int pn = KB / jn;
    const int tiles = (t + pn - 1) / pn;
    const int nhl = KB / (pn * (jn / vec));
    // Heads are split over workgroups only as far as the positions leave the
    // chip short of four workgroups a compute unit: each group evaluates the
    // angles again.
    const int most = (heads + nhl - 1) / nhl;
    const int groups = std::max(1, std::min(most, (1024 + tiles - 1) / tiles));
    const int hpb = (heads + groups * nhl - 1) / (groups * nhl) * nhl;
    const dim3 g((unsigned)((long)tiles * groups * chunks)), b(KB);
#define ROPE(V, H, G) \
    hipLaunchKernelGGL((rope_kernel<V, H>), G, b, 0, st, x, off, div, t, heads, hd, theta, first, pn, jn, tiles, groups, hpb)
    if (vec == 4 && hd == 128) ROPE(4, 128, dim3(tiles, groups));
    else if (vec == 4 && hd == 64) ROPE(4, 64, dim3(tiles, groups));
    else if (vec == 4) ROPE(4, 0, g);
    else ROPE(1, 0, g);
#undef ROPE
    return hipGetLastError();
}

template <typename T>
static hipError_t launch_append_as(const float* src, T* dst, int tr, int n, int kv, int hd, int cap, int past,
                                   hipStream_t st) {
    const long d = (long)kv * hd, tot = n * d;
    const bool in16 = aligned16(src) && d % 4 == 0;
    if (!tr && in16 && hd % 8 == 0 && aligned16(dst) && tot / 8 <= 0x7fffffffL) {
        hipLaunchKernelGGL((append_k8_kernel<T>), dim3(nblk(tot / 8)), dim3(KB), 0, st, src, dst, (unsigned)(tot / 8),
                           (unsigned)(d / 8), (unsigned)(hd / 8), cap, past);
        return hipGetLastError();
    }
    // The tiles pay from about a quarter of one in positions (below, the flat
    // form's scattered stores are as few).
    if (tr && in16 && d % AT_D == 0 && d / AT_D <= 65535 && n >= AT_P / 4) {
        const int wide = cap % 4 == 0 && reinterpret_cast<uintptr_t>(dst) % (4 * sizeof(T)) == 0;
        const dim3 g((unsigned)((past + n - 1) / AT_P - past / AT_P + 1), (unsigned)(d / AT_D));
        hipLaunchKernelGGL((append_vt_kernel<T>), g, dim3(KB), 0, st, src, dst, n, (int)d, cap, past, wide);
        return hipGetLastError();
    }
    const dim3 g(nblk(tot)), b(KB);
    if (tr) hipLaunchKernelGGL((append_kernel<T, true>), g, b, 0, st, src, dst, n, kv, hd, cap, past);
    else hipLaunchKernelGGL((append_kernel<T, false>), g, b, 0, st, src, dst, n, kv, hd, cap, past);
    return hipGetLastError();
}

hipError_t launch_append(const float* src, long src_off, void* dst, int f16, int tr, int n, int kv, int hd, int cap,
                         int past, hipStream_t st) {
    if ((long)n * kv * hd == 0) return hipSuccess;
    if (f16) return launch_append_as(src + src_off, (uint16_t*)dst, tr, n, kv, hd, cap, past, st);
    return launch_append_as(src + src_off, (float*)dst, tr, n, kv, hd, cap, past, st);
}

hipError_t launch_rope_cache_f16(float* q, long q_off, const float* k, long k_off, const float* v, long v_off,
                                 const float* div, int heads, int kv, int hd, float theta, int pos, uint16_t* kc,
                                 uint16_t* vc, int cap, hipStream_t st) {
    const long n = (long)heads * (hd / 2) + (long)kv * (hd / 2) + (long)kv * hd;
#define RC(H)                                                                                                    \
    hipLaunchKernelGGL((rope_cache_f16_kernel<H>), dim3(nblk(n)), dim3(KB), 0, st, q + q_off, k + k_off, v + v_off, div, \
                       heads, kv, hd, theta, pos, kc, vc, cap)
    if (hd == 128) RC(128);
    else if (hd == 64) RC(64);
    else RC(0);
#undef RC
    return hipGetLastError();
}

hipError_t launch_grow(const void* src, void* dst, int esz, int rows, int len, int ss, int ds, hipStream_t st) {
    const long n = (long)rows * len;
    if (n == 0) return hipSuccess;
    if (esz == 2) hipLaunchKernelGGL((grow_kernel<uint16_t>), dim3(nblk(n)), dim3(KB), 0, st, (const uint16_t*)src, (uint16_t*)dst, rows, len, ss, ds);
    else if (esz == 1) hipLaunchKernelGGL((grow_kernel<int8_t>), dim3(nblk(n)), dim3(KB), 0, st, (const int8_t*)src, (int8_t*)dst, rows, len, ss, ds);
    else hipLaunchKernelGGL((grow_kernel<float>), dim3(nblk(n)), dim3(KB), 0, st, (const float*)src, (float*)dst, rows, len, ss, ds);
    return hipGetLastError();
}

hipError_t launch_append_q8(const float* k, long k_off, const float* v, long v_off, char* cache, int slot, int n,
                            int kv, int hd, int cap, int past, hipStream_t st) {
    const long tot = (long)n * kv * hd;
    if (tot == 0) return hipSuccess;
    const int b0 = past / 32;
    const long units = (long)((past + n - 1) / 32 - b0 + 1) * kv * (hd / 16);
    // As launch_append_t16, from half as many elements (there are two areas):
    // 60 rows of 8 x 128, 3.59 us in chunks and 3.44 flat; 173 rows, 3.64 and 3.87.
    const long wgs = chunk_wgs(units, (long)Edges(past, n).count() * kv * hd);
    if (tot >= 1L << 17 && aligned16(k + k_off) && aligned16(cache) && hd % 64 == 0 && wgs <= CHUNK_WGS) {
        const dim3 g((unsigned)wgs);
        hipLaunchKernelGGL(append_q8_chunks_kernel, g, dim3(KB), 0, st, k + k_off, v + v_off, cache, slot, n, kv, hd, tiled_nblk(cap), past, (int)units, b0);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(append_q8_kernel, dim3(nblk(tot)), dim3(KB), 0, st, k, k_off, v, v_off, cache, slot, n, kv, hd,
                       cap, past);
    return hipGetLastError();
}

hipError_t launch_rope_cache_q8(float* q, long q_off, const float* k, long k_off, const float* v, long v_off,
                                const float* div, int heads, int kv, int hd, float theta, int pos, char* cache,
                                int slot, int cap, hipStream_t st) {
    const unsigned qb = nblk((long)heads * (hd / 2));
    const unsigned kb = nblk(2L * kv * hd);
#define RC(H)                                                                                                    \
    hipLaunchKernelGGL((rope_cache_q8_kernel<H>), dim3(qb + kb), dim3(KB), 0, st, q + q_off, k + k_off, v + v_off, div, \
                       heads, kv, hd, theta, pos, cache, slot, cap)
    if (hd == 128) RC(128);
    else if (hd == 64) RC(64);
    else RC(0);
#undef RC
    return hipGetLastError();
}

hipError_t launch_append_t16(const float* src, long src_off, uint16_t* cache, int n, int kv, int hd, int cap,
                             int past, int value, hipStream_t st) {
    const long tot = (long)n * kv * hd;
    if (tot == 0) return hipSuccess;
    const int b0 = past / 32;
    const long units = (long)((past + n - 1) / 32 - b0 + 1) * kv * (value ? hd / 64 : hd / 16);
    // Whole chunks once the flat form would take about 1024 workgroups (V) or
    // from two rows on (K, whose chunks are one key's): 173 rows of 8 x 128, V
    // 2.66 us in chunks and 2.57 flat; 300 rows, 3.17 and 3.31; K even at 29.
    const long wgs = chunk_wgs(units, value ? (long)Edges(past, n).count() * kv * hd : 0);
    if ((value ? tot >= 1L << 18 : n > 1) && aligned16(src + src_off) && aligned16(cache) && hd % 64 == 0 && wgs <= CHUNK_WGS) {
        const dim3 g((unsigned)wgs);
        if (value) hipLaunchKernelGGL((append_t16_chunks_kernel<true>), g, dim3(KB), 0, st, src + src_off, cache, n, kv, hd, tiled_nblk(cap), past, (int)units, b0);
        else hipLaunchKernelGGL((append_t16_chunks_kernel<false>), g, dim3(KB), 0, st, src + src_off, cache, n, kv, hd, tiled_nblk(cap), past, (int)units, b0);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(append_t16_kernel, dim3(nblk(tot)), dim3(KB), 0, st, src, src_off, cache, n, kv, hd, cap,
                       past, value);
    return hipGetLastError();
}

hipError_t launch_rope_cache_t16(float* q, long q_off, const float* k, long k_off, const float* v, long v_off,
                                 const float* div, int heads, int kv, int hd, float theta, int pos, uint16_t* cache,
                                 int cap, hipStream_t st) {
    const long n = (long)heads * (hd / 2) + (long)kv * (hd / 2) + (long)kv * hd;
#define RC(H)                                                                                                    \
    hipLaunchKernelGGL((rope_cache_t16_kernel<H>), dim3(nblk(n)), dim3(KB), 0, st, q + q_off, k + k_off, v + v_off, div, \
                       heads, kv, hd, theta, pos, cache, cap)
    if (hd == 128) RC(128);
    else if (hd == 64) RC(64);
    else RC(0);
#undef RC
    return hipGetLastError();
}

hipError_t launch_ref_to_t16(const uint16_t* k, const uint16_t* v, uint16_t* cache, int kv, int hd, int cap, int live,
                             int tcap, hipStream_t st) {
    const long n = 2L * kv * ((live + 31) / 32) * 32 * hd;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(ref_to_t16_kernel, dim3(nblk(n)), dim3(KB), 0, st, k, v, cache, kv, hd, cap, live, tcap);
    return hipGetLastError();
}

}  // namespace llmtie
