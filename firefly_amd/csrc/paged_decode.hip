// paged_decode.hip - PagedAttention decode for gfx950: GQA-shared KV reads, split-K over the context, online
// softmax, and a merge pass.
//
// Reference semantics: paged_attention_kernel (src/kernels/attention.cu:291-447).  The reference runs one
// 128-thread block per (query head, sequence), so every query head of a GQA group re-reads the same KV head, and
// a long context is walked serially by one block.  Here one 256-thread workgroup owns a (chunk, kv_head,
// sequence) work item: it loads the G = Hq/Hkv query vectors of the group once, reads each K/V page slice once
// for all of them, and writes either the final output (rows that fit in one chunk) or an unnormalised partial
// state (m, l, acc) that paged_decode_merge combines.
//
// Lane layout: head_dim/8 lanes per token (one 8-element, 16-byte chunk each for 16-bit KV), so a wave64 covers
// 64/(D/8) tokens per step and the workgroup 256/(D/8).  Head dims other than 64, 128 and 256 (multiples of 8 up
// to 128, which the reference's decode takes) run with 16 lanes per token, those past head_dim/8 idle.  Each token slot keeps its own online-softmax state in
// registers; the slots are merged with cross-lane shuffles inside a wave and through LDS across waves.
// The softmax runs in base 2 with log2(e) folded into the score scale, against a reference maximum that moves only
// when a score passes it by 2^8.  A token's dot product crosses its lanes with DPP steps (no LDS), and each loop
// trip issues the loads of several token groups (and the next trip's block-table entries) before using them: the
// kernel is bound by memory latency, not by its arithmetic.
#include "ffkv_device.h"
#include "ffkv_internal.h"

namespace ffkv
{

namespace
{

#ifndef FFKV_GENERIC_U16
#define FFKV_GENERIC_U16 4  // token groups per loop trip: other caches
#endif
#ifndef FFKV_GENERIC_U32
#define FFKV_GENERIC_U32 2  // token groups per loop trip: fp32 caches (a raw row takes twice the registers)
#endif

constexpr float kNegBig = -1e30f;  // finite "minus infinity" seed, as in attention.cu:323

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

using u32x4 = uint32_t __attribute__((ext_vector_type(4)));

// Dims held by a lane of a D-dim row, the same for q, K, V and the output: 8 consecutive ones (16 bytes of a 16-bit
// cache).  A lane's 8 fp32 values are two 16-byte loads, so they come from the row's two halves, four from each:
// either load then covers whole lines of consecutive lanes, where 8 consecutive dims would have both loads touch
// every line.
template <int CT>
__device__ __forceinline__ int lane_dim(int D, int lane, int i)
{
    return CT == F32 ? (i >> 2) * (D >> 1) + 4 * lane + (i & 3) : 8 * lane + i;
}

template <int CT, bool NT>
__device__ __forceinline__ void load_row8(const void* base, size_t row, int D, int lane, Raw8& r)
{
    if constexpr (CT == F32)
    {
        const float* p = static_cast<const float*>(base) + row * D;
#pragma unroll
        for (int h = 0; h < 2; ++h)
        {
            const u32x4* s = reinterpret_cast<const u32x4*>(p + lane_dim<CT>(D, lane, 4 * h));
            const u32x4  w = NT ? __builtin_nontemporal_load(s) : *s;
#pragma unroll
            for (int i = 0; i < 4; ++i) r.w[4 * h + i] = w[i];
        }
    }
    else
    {
        load_raw8<CT>(base, row * D + lane * 8, r);
    }
}

__device__ __forceinline__ int row_tokens(const DecodeArgs& a, int b)
{
    int64_t L = static_cast<int64_t>(a.context_lens[b]) + 1;  // +1: the token appended this step (:320)
    if (L > a.cap_tokens) L = a.cap_tokens;
    return L < 0 ? 0 : static_cast<int>(L);
}

}  // namespace

// DT: head_dim, or 0 for a runtime head_dim (a multiple of 8 up to 8 * LPT); LPT: lanes per token, a power of two
// (DT / 8 when DT is given).  Lanes past head_dim / 8 hold zeros and store nothing.
template <int CT, int DT, int LPT, int GP>
__global__ __launch_bounds__(256) void paged_decode_generic(DecodeArgs a)
{
    static_assert(DT == 0 || DT == 8 * LPT, "a given head_dim has head_dim / 8 lanes per token");
    constexpr int TPI = 256 / LPT; // token slots per workgroup
    constexpr int WAVES = 4;
    constexpr int DMAX = 8 * LPT;
    const int     D = DT != 0 ? DT : a.head_dim;

    const int chunk_id = blockIdx.x;
    const int kvh = blockIdx.y;
    const int b = blockIdx.z;
    const int tid = threadIdx.x;
    const int lane = tid % LPT;
    const int slot = tid / LPT;
    const int wave = tid / 64;
    const bool act = DT != 0 || lane * 8 < D;  // this lane holds dims of the head

    const int L = row_tokens(a, b);
    const int nch = (L + a.chunk - 1) / a.chunk;
    if (chunk_id >= nch && !(chunk_id == 0 && nch == 0)) return;  // uniform over the workgroup
    const int begin = chunk_id * a.chunk;
    const int end = min(begin + a.chunk, L);
    const int G = a.group;

    const int32_t* table = a.block_table + static_cast<int64_t>(b) * a.max_blocks;
    // the chunk's first page in this row and in one of the 256 rows around it, a thread each (see `once`)
    int first = -1, other = -2;
    if constexpr (CT == F32)
    {
        const int r = max(0, min(b - 128, a.batch - 256)) + tid;
        if (begin < end)
        {
            first = table[begin >> 4];
            if (r != b && r < a.batch) other = a.block_table[static_cast<int64_t>(r) * a.max_blocks + (begin >> 4)];
        }
    }

    float q[GP][8];
#pragma unroll
    for (int g = 0; g < GP; ++g)
    {
        if (g < G && act)
        {
            const size_t qb = (static_cast<size_t>(b) * a.num_heads + kvh * G + g) * D;
            if constexpr (CT == F32)
            {
                load_act4(a.q, a.qo_dtype, qb + lane_dim<CT>(D, lane, 0), q[g]);
                load_act4(a.q, a.qo_dtype, qb + lane_dim<CT>(D, lane, 4), q[g] + 4);
            }
            else
                load_act8(a.q, a.qo_dtype, qb + lane * 8, q[g]);
        }
        else
#pragma unroll
            for (int i = 0; i < 8; ++i) q[g][i] = 0.0f;
    }

    float m[GP], l[GP], acc[GP][8];
#pragma unroll
    for (int g = 0; g < GP; ++g)
    {
        m[g] = kNegBig;
        l[g] = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[g][i] = 0.0f;
    }

    // fp32 pages are read past the caches, unless another row holds the chunk's first page too (a shared prefix, which the
    // rows' workgroups then read from the caches).  32 rows of 512 to 4096 tokens at 32/8 heads take 128 us per call with
    // plain loads and 113 with these, 120 rows over a 2048-token prefix 188 us with plain loads and 275 with these.  (Four
    // token groups per trip gain another 1 % on the former and cost the latter 10 %: fewer waves fit.)  Any of the 256
    // rows around this one counts, a thread each: rows over two or ten prefixes in turn, no two neighbours alike, took 296
    // and 395 us where only the rows on either side were looked at, 194 and 357 now (all plain: 204 and 360).
    bool once = CT == F32;
    if constexpr (CT == F32) once = __syncthreads_or(first == other) == 0;

    // U consecutive token groups per loop trip: their table entries, then all their K / V loads, go out before
    // any of them is used, so U times the bytes of one group are in flight per wave (none extra for the 16-head
    // groups, which already fill the registers).  The table entries of the next trip are requested while this trip's
    // tokens are computed.
    // ALWAYS: tokens of no page, and lanes past the head, load too (from page 0, the token's first dims) and are left out
    // where they would count.  Behind a branch the wait for the first group's K is, as far as the compiler can tell, one for
    // nearly all loads, so that nothing is computed while they are on their way: with eight heads per KV head, where
    // computing takes as long as loading, 32 rows of 512 to 4096 fp32 tokens at 64/8 heads 172.9 -> 165.7 us, 36 of 6600 to
    // 12500 at head_dim 80 590 -> 555; with four heads of 128 dims 111.3 -> 112.1, with one at head_dim 72 (fp8) 36.4 -> 36.9.
    constexpr bool ALWAYS = GP >= 8 || (DT == 0 && GP >= 4);
    const int      stop = ALWAYS && a.num_blocks <= 0 ? begin : end;  // without a page there is nothing to load from
    auto stream = [&]<int U, bool NT>()
    {
        auto load_phys = [&](int base, int (&ph)[U])
        {
#pragma unroll
            for (int u = 0; u < U; ++u)
            {
                const int j = base + u * TPI + slot;
                ph[u] = j < end ? table[j >> 4] : -1;
            }
        };
        int phys[U];
        load_phys(begin, phys);
        for (int base = begin; base < stop; base += U * TPI)
        {
            bool   valid[U];
            size_t row[U];
            float  ks[U], vs[U];  // int8: the tokens' scales
#pragma unroll
            for (int u = 0; u < U; ++u)
            {
                const int j = base + u * TPI + slot;
                valid[u] = j < end && phys[u] >= 0 && phys[u] < a.num_blocks;
                row[u] = (static_cast<size_t>(valid[u] ? phys[u] : 0) * kBlockSize + (j & 15)) * a.num_kv_heads + kvh;
            }
            Raw8 kr[U], vr[U];
#pragma unroll
            for (int u = 0; u < U; ++u)
            {
                ks[u] = vs[u] = 1.0f;
                if (ALWAYS || (valid[u] && act))
                {
                    const int ln = act ? lane : 0;
                    load_row8<CT, NT>(a.k_cache, row[u], D, ln, kr[u]);
                    load_row8<CT, NT>(a.v_cache, row[u], D, ln, vr[u]);
                    if constexpr (CT == I8)
                    {
                        ks[u] = a.k_scale[row[u]];
                        vs[u] = a.v_scale[row[u]];
                    }
                }
                else
                {
                    kr[u] = Raw8{};
                    vr[u] = Raw8{};
                }
            }
            load_phys(base + U * TPI, phys);
#pragma unroll
            for (int u = 0; u < U; ++u)
            {
                float k[8];
                unpack8<CT>(kr[u], k);
                if constexpr (ALWAYS && DT == 0)
#pragma unroll
                    for (int i = 0; i < 8; ++i) k[i] = act ? k[i] : 0.0f;
                if constexpr (CT == I8 || CT == FP8)
                {
                    const float sk = CT == I8 ? ks[u] : a.k_scale[kvh];
#pragma unroll
                    for (int i = 0; i < 8; ++i) k[i] *= sk;
                }
                float s[GP];
#pragma unroll
                for (int g = 0; g < GP; ++g)
                {
                    float d = 0.0f;
#pragma unroll
                    for (int i = 0; i < 8; ++i) d = __builtin_fmaf(q[g][i], k[i], d);
                    s[g] = d;
                }
                // every lane takes part in the sums (DPP lane steps); a token's lanes are a contiguous, aligned group
#pragma unroll
                for (int g = 0; g < GP; ++g) s[g] = group_sum<LPT>(s[g]);

                // Online softmax with a lazy reference: m moves (and l, acc are rescaled) only when a score exceeds it
                // by more than 8 (log2 units), so p = 2^(s - m) < 2^8 and most tokens only add p and p * v.
                if (valid[u])
                {
                    float v[8];  // unpacked only now: fewer registers live across the dot products and sums
                    unpack8<CT>(vr[u], v);
                    if constexpr (CT == I8 || CT == FP8)
                    {
                        const float sv = CT == I8 ? vs[u] : a.v_scale[kvh];
#pragma unroll
                        for (int i = 0; i < 8; ++i) v[i] *= sv;
                    }
#pragma unroll
                    for (int g = 0; g < GP; ++g)
                    {
                        const float sg = s[g] * a.scale_log2;
                        if (sg > m[g] + 8.0f)
                        {
                            const float alpha = fast_exp2(m[g] - sg);  // 0 for the slot's first token
                            l[g] *= alpha;
#pragma unroll
                            for (int i = 0; i < 8; ++i) acc[g][i] *= alpha;
                            m[g] = sg;
                        }
                        const float p = fast_exp2(sg - m[g]);
                        l[g] += p;
#pragma unroll
                        for (int i = 0; i < 8; ++i) acc[g][i] = __builtin_fmaf(p, v[i], acc[g][i]);
                    }
                }
            }
        }
    };
    constexpr int U = GP >= 16 ? 1 : (CT == F32 ? FFKV_GENERIC_U32 : FFKV_GENERIC_U16);
    if (CT == F32 && once)
        stream.template operator()<U, CT == F32>();
    else
        stream.template operator()<U, false>();

    // merge the token slots of this wave (lanes lane, lane+LPT, ... hold the same dims)
#pragma unroll
    for (int off = LPT; off < 64; off <<= 1)
    {
#pragma unroll
        for (int g = 0; g < GP; ++g)
        {
            const float mo = shfl_xor(m[g], off);
            const float lo = shfl_xor(l[g], off);
            const float mn = fmaxf(m[g], mo);
            const float a1 = fast_exp2(m[g] - mn);
            const float a2 = fast_exp2(mo - mn);
            l[g] = l[g] * a1 + lo * a2;
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[g][i] = acc[g][i] * a1 + shfl_xor(acc[g][i], off) * a2;
            m[g] = mn;
        }
    }

    // merge the waves through LDS, one wave at a time
    __shared__ float s_acc[GP][DMAX];
    __shared__ float s_m[GP];
    __shared__ float s_l[GP];
    const bool holder = (tid % 64) < LPT && act;
    for (int w = 0; w < WAVES; ++w)
    {
        if (wave == w && holder)
        {
#pragma unroll
            for (int g = 0; g < GP; ++g)
            {
                if (w == 0)
                {
#pragma unroll
                    for (int i = 0; i < 8; ++i) s_acc[g][lane_dim<CT>(D, lane, i)] = acc[g][i];
                    if (lane == 0)
                    {
                        s_m[g] = m[g];
                        s_l[g] = l[g];
                    }
                }
                else
                {
                    const float mo = s_m[g];
                    const float lo = s_l[g];
                    const float mn = fmaxf(m[g], mo);
                    const float a1 = fast_exp2(m[g] - mn);
                    const float a2 = fast_exp2(mo - mn);
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                    {
                        float& o = s_acc[g][lane_dim<CT>(D, lane, i)];
                        o = acc[g][i] * a1 + o * a2;
                    }
                    // all holder lanes read s_m/s_l before lane 0 overwrites them: same wave, lockstep
                    __builtin_amdgcn_wave_barrier();
                    if (lane == 0)
                    {
                        s_m[g] = mn;
                        s_l[g] = l[g] * a1 + lo * a2;
                    }
                }
            }
        }
        __syncthreads();
    }

    const int     hq0 = kvh * G;
    const bool    single = nch <= 1;
    const int64_t ml_base = (static_cast<int64_t>(b) * a.num_heads + hq0) * a.max_chunks + chunk_id;
    for (int idx = tid; idx < G * D; idx += 256)
    {
        const int   g = idx / D;
        const int   d = idx % D;
        const float acc_v = s_acc[g][d];
        if (single)
        {
            const float lsum = s_l[g];
            store_act1(a.out, a.qo_dtype, (static_cast<size_t>(b) * a.num_heads + hq0 + g) * D + d,
                       lsum == 0.0f ? 0.0f : acc_v / lsum);
        }
        else
        {
            const int64_t pi = ml_base + static_cast<int64_t>(g) * a.max_chunks;
            a.ws_acc[pi * D + d] = acc_v;
            if (d == 0)
            {
                a.ws_ml[2 * pi] = s_m[g];
                a.ws_ml[2 * pi + 1] = s_l[g];
            }
        }
    }
}

// Combine the chunk partials of rows that needed more than one chunk: thread k of row b's workgroups folds dims
// 4 (k % (D/4)) .. + 3 of head k / (D/4) over the row's chunks, the loads of MF chunks in flight together (one
// workgroup per head, its threads walking the chunks three times with one load in flight, took 11.6 us on 32 rows of
// 512 to 4096 tokens; this takes 5.0).
__global__ __launch_bounds__(256) void paged_decode_merge(DecodeArgs a)
{
    constexpr int MF = 8;
    const int     D = a.head_dim;
    const int     b = blockIdx.x;
    const int     k = static_cast<int>(blockIdx.y) * 256 + static_cast<int>(threadIdx.x);
    const int     L = row_tokens(a, b);
    const int     nch = (L + a.chunk - 1) / a.chunk;
    if (nch <= 1 || k >= a.num_heads * (D / 4)) return;
    const int     h = k / (D / 4);
    const int     d4 = (k - h * (D / 4)) * 4;
    const int64_t base = (static_cast<int64_t>(b) * a.num_heads + h) * a.max_chunks;
    float         m = kNegBig, l = 0.0f, o[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int c0 = 0; c0 < nch; c0 += MF)
    {
        float2 t[MF];
        float4 x[MF];
        float  mn = m;
#pragma unroll
        for (int f = 0; f < MF; ++f)
        {
            t[f] = make_float2(kNegBig, 0.0f);
            x[f] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (c0 + f < nch)
            {
                t[f] = *reinterpret_cast<const float2*>(a.ws_ml + 2 * (base + c0 + f));
                x[f] = *reinterpret_cast<const float4*>(a.ws_acc + (base + c0 + f) * D + d4);
            }
        }
#pragma unroll
        for (int f = 0; f < MF; ++f) mn = fmaxf(mn, t[f].x);
        const float wa = fast_exp2(m - mn);
        l *= wa;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] *= wa;
#pragma unroll
        for (int f = 0; f < MF; ++f)
        {
            const float w = fast_exp2(t[f].x - mn);
            l += t[f].y * w;
            o[0] += x[f].x * w, o[1] += x[f].y * w, o[2] += x[f].z * w, o[3] += x[f].w * w;
        }
        m = mn;
    }
    const float  inv = softmax_inv(l);
    const size_t ob = (static_cast<size_t>(b) * a.num_heads + h) * D + d4;
#pragma unroll
    for (int i = 0; i < 4; ++i) store_act1(a.out, a.qo_dtype, ob + i, o[i] * inv);
}

namespace
{

template <int CT, int DT, int LPT, int GP>
hipError_t launch3(const DecodeArgs& a, hipStream_t stream)
{
    dim3 grid(static_cast<unsigned>(a.max_chunks), static_cast<unsigned>(a.num_kv_heads),
              static_cast<unsigned>(a.batch));
    hipLaunchKernelGGL((paged_decode_generic<CT, DT, LPT, GP>), grid, dim3(256), 0, stream, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || a.max_chunks <= 1) return e;
    hipLaunchKernelGGL(paged_decode_merge,
                       dim3(static_cast<unsigned>(a.batch),
                            static_cast<unsigned>((a.num_heads * (a.head_dim / 4) + 255) / 256)),
                       dim3(256), 0, stream, a);
    return hipGetLastError();
}

template <int CT, int DT, int LPT>
hipError_t launch2(const DecodeArgs& a, hipStream_t stream)
{
    if (a.group <= 1) return launch3<CT, DT, LPT, 1>(a, stream);
    if (a.group <= 2) return launch3<CT, DT, LPT, 2>(a, stream);
    if (a.group <= 4) return launch3<CT, DT, LPT, 4>(a, stream);
    if (a.group <= 8) return launch3<CT, DT, LPT, 8>(a, stream);
    return launch3<CT, DT, LPT, 16>(a, stream);
}

template <int CT>
hipError_t launch1(const DecodeArgs& a, hipStream_t stream)
{
    switch (a.head_dim)
    {
        case 64:
            return launch2<CT, 64, 8>(a, stream);
        case 128:
            return launch2<CT, 128, 16>(a, stream);
        case 256:
            return launch2<CT, 256, 32>(a, stream);
        default:  // any other multiple of 8 up to 128: 16 lanes per token, those past head_dim / 8 idle
            return launch2<CT, 0, 16>(a, stream);
    }
}

}  // namespace

hipError_t launch_decode(const DecodeArgs& a, hipStream_t stream)
{
    switch (a.cache_dtype)
    {
        case F32:
            return launch1<F32>(a, stream);
        case F16:
            return launch1<F16>(a, stream);
        case BF16:
            return launch1<BF16>(a, stream);
        case I8:
            return launch1<I8>(a, stream);
        default:
            return launch1<FP8>(a, stream);
    }
}

}  // namespace ffkv
