// Matrix-pipe ceiling probe for gfx950 (MI355X): a loop of nothing but the GEMM kernels' MFMA, in the GEMM's
// register pattern and order, with every operand held in registers: no LDS, no memory.  One workgroup of four wavefronts
// per compute unit (one per SIMD), like the 256x256 GEMM tile.  Two forms: v_mfma_f32_32x32x16_bf16 (a wavefront
// owns a 4 x 4 grid of 32x32 accumulators and multiplies four A fragments with four B fragments per k16 step) and
// v_mfma_f32_16x16x32_bf16 (8 x 8 accumulators of 16x16, eight fragments of each operand per k32 step).  Both in the order of
// the GEMM's pipelines on that MFMA: row after row the former, the latter as RollPipe::quarter, or in one of three others for comparison.
//
// The operands of consecutive k16 steps rotate over SETS register-resident fragment sets filled
// with a pattern: zeros, one constant, or N(0, 0.02)-like pseudo-random bf16 values.  The rate
// the loop sustains with random operands is what the matrix pipes deliver under the board's power
// limit when the data toggles; with constant operands it is the limit of the pipes themselves.
#include "common.h"

namespace syn {

typedef unsigned int u32x4_probe_t __attribute__((ext_vector_type(4)));

constexpr int kProbeSets = 4;

__device__ __forceinline__ unsigned probe_hash(unsigned x) {
    x ^= x >> 16;
    x *= 0x7feb352du;
    x ^= x >> 15;
    x *= 0x846ca68bu;
    x ^= x >> 16;
    return x;
}

// pattern 0: zeros; 1: every element 1.0; 2: pseudo-random, roughly N(0, 0.02) (sum of four uniforms)
__device__ __forceinline__ bf16x8_t probe_fragment(int pattern, unsigned seed) {
    bf16x8_t f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float v = 0.f;
        if (pattern == 1) v = 1.0f;
        if (pattern == 2) {
            const unsigned h = probe_hash(seed * 8u + e);
            const float u = (float)(h & 0xff) + (float)((h >> 8) & 0xff) + (float)((h >> 16) & 0xff) + (float)(h >> 24);
            v = (u - 510.f) * (0.02f / 147.8f);      // variance of the sum of four U{0..255}: 4 * 5461.25
        }
        f[e] = (__bf16)v;
    }
    return f;
}

__global__ void __launch_bounds__(256) mfma_rate_kernel(float* sink, int iters, int pattern) {
    f32x16_t acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    bf16x8_t fa[kProbeSets][4], fb[kProbeSets][4];
    const unsigned me = blockIdx.x * 256u + threadIdx.x;
#pragma unroll
    for (int s = 0; s < kProbeSets; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            fa[s][i] = probe_fragment(pattern, (me * kProbeSets + s) * 8u + i);
            fb[s][i] = probe_fragment(pattern, (me * kProbeSets + s) * 8u + 4u + i);
        }
    for (int it = 0; it < iters; ++it) {
#pragma unroll
        for (int s = 0; s < kProbeSets; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[s][j], fa[s][i], acc[i][j], 0, 0, 0);
    }
    float total = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) total += acc[i][j][0] + acc[i][j][7];
    sink[me] = total;
}

// How the 16x16x32 MFMAs of a k32 step follow each other.  What changes from one to the next is what switches:
//   kOrderPairs     the GEMM's: two columns of accumulators at a time, down the rows and up again: A and B in turn
//   kOrderRows      row after row: B, and A too at the end of a row
//   kOrderToAndFro  every other row backwards: B, or A at the end of a row
//   kOrderDiagonal  both every time
constexpr int kOrderPairs = 0, kOrderRows = 1, kOrderToAndFro = 2, kOrderDiagonal = 3;

// the same on 16x16x32 MFMAs: 128 per round, the flop of 64 of the larger ones.  The accumulators are named as AGPR
// tuples in inline assembly, as in the GEMM's K loop.
template <int ORDER>
__global__ void __launch_bounds__(256) mfma16_rate_kernel(float* sink, int iters, int pattern) {
    typedef float f32x4_probe_t __attribute__((ext_vector_type(4)));
    f32x4_probe_t acc[8][8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_probe_t{0.f, 0.f, 0.f, 0.f};
    bf16x8_t fa[2][8], fb[2][8];
    const unsigned me = blockIdx.x * 256u + threadIdx.x;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            fa[s][i] = probe_fragment(pattern, (me * 2u + s) * 16u + i);
            fb[s][i] = probe_fragment(pattern, (me * 2u + s) * 16u + 8u + i);
        }
    for (int it = 0; it < iters; ++it) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int g = 0; g < 64; ++g) {
                int i = g / 8, j = g % 8;
                if (ORDER == kOrderPairs) {
                    // a half of four rows against all columns, then the other
                    const int h = g % 32, row = h % 8 / 2;
                    i = 4 * (g / 32) + (h / 8 % 2 == 0 ? row : 3 - row);
                    j = 2 * (h / 8) + (h % 2 ^ row % 2);
                } else if (ORDER == kOrderToAndFro) {
                    j = i % 2 == 0 ? j : 7 - j;
                } else if (ORDER == kOrderDiagonal) {
                    j = g % 8;
                    i = (g / 8 + g) % 8;
                }
                asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(fb[s][j]), "v"(fa[s][i]));
            }
    }
    // the compiler adds no wait states behind assembly MFMAs: a matrix op of N passes needs N + 3 of them (at
    // most 19) before a vector instruction may read its result
    asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
    float total = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) total += acc[i][j][0] + acc[i][j][3];
    sink[me] = total;
}

// HBM read ceiling probe: `STREAMS` read streams `stride_vecs` 16-byte groups apart, walked in the chunked
// reduce's access pattern - 256 lanes, four groups per lane and pass, every load of a pass issued
// before the first is used, non-temporal - with an exclusive-or in place of the adds and no result
// stream.  What it sustains is what the memory system gives that pattern of reads.
constexpr int kStreamThreads = 256;
constexpr int kStreamVecs = 4;

template <int STREAMS>
__global__ void __launch_bounds__(kStreamThreads)
read_streams_kernel(const u32x4_probe_t* __restrict__ base, int64_t stride_vecs, int64_t stream_vecs,
                    u32x4_probe_t* __restrict__ sink) {
    constexpr int64_t kGroup = (int64_t)kStreamThreads * kStreamVecs;
    u32x4_probe_t mix = {0u, 0u, 0u, 0u};
    for (int64_t g0 = (int64_t)blockIdx.x * kGroup; g0 + kGroup <= stream_vecs; g0 += (int64_t)gridDim.x * kGroup) {
        u32x4_probe_t parts[kStreamVecs][STREAMS];
#pragma unroll
        for (int u = 0; u < kStreamVecs; ++u)
#pragma unroll
            for (int i = 0; i < STREAMS; ++i)
                parts[u][i] = __builtin_nontemporal_load(base + (int64_t)i * stride_vecs + g0 + threadIdx.x + u * kStreamThreads);
#pragma unroll
        for (int u = 0; u < kStreamVecs; ++u)
#pragma unroll
            for (int i = 0; i < STREAMS; ++i) mix ^= parts[u][i];
    }
    // keeps the loads alive; a lane whose words happen to cancel leaves its note in the sink
    if ((mix.x ^ mix.y ^ mix.z ^ mix.w) == 0x9e3779b9u) sink[blockIdx.x] = mix;
}


// ---- the paired attention kernel's slot, piece by piece -------------------------------------------------------
// A workgroup of eight wavefronts, two per SIMD, like attn_pair_kernel.  Per iteration ("slot") wavefronts 0-3
// run that kernel's matrix products - 32 MFMAs 32x32x16 fed by transposing 8-byte LDS reads (P.V) and 32 fed by
// 16-byte LDS reads (Q.K), the reads two steps ahead of their MFMA, same addresses and swizzles - and wavefronts
// 4-7 one softmax pass over 64 scores per lane (maximum, exponentials, sum, conversion to 16-bit pairs).  Every
// piece can be switched off, so that what each costs beside the others is measured and not inferred:
//   kSlotProducts / kSlotSoftmax   which half of the workgroup works (the other only joins the barriers)
//   kSlotLds        the products' K and V fragments come from LDS (else the loop runs on register operands)
//   kSlotFills      every wavefront issues four 1 KB LDS-DMA fills per slot (the kernel's 64 KB per two slots)
//   kSlotPrefetch   the first fragments of the next phase are asked for in the tail of the previous one
//   kSlotRandom     LDS and the register operands hold pseudo-random values instead of one constant
//   kSlotPrivate    a workgroup's fills read a region of its own (misses in the L2); else every workgroup reads the
//                   same 32 KB piece per slot - one miss per XCD, then L2 hits, like programs that walk one head's K, V
//   kSlotNarrow     every 32x32x16 MFMA is replaced by two 16x16x32 MFMAs that share its A operand (the same flop,
//                   the same LDS reads, half of the accumulator registers): the form attn_pair_kernel uses, whose
//                   32 q rows per wavefront are two halves of 16
// A slot ends like the kernel's: wait for the wavefront's own LDS reads (and fills), then the barrier.
constexpr int kSlotProducts = 1, kSlotSoftmax = 2, kSlotLds = 4, kSlotFills = 8, kSlotPrefetch = 16, kSlotRandom = 32,
              kSlotPrivate = 64, kSlotNarrow = 128;
constexpr int kSlotRowBytes = 256, kSlotBlockBytes = 32768;
typedef short slot_s16x4_t __attribute__((ext_vector_type(4)));
typedef short slot_s16x8_t __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) slot_s16x4_t* slot_lds_s16x4_ptr;
typedef __attribute__((address_space(3))) void* slot_lds_ptr;
typedef const __attribute__((address_space(1))) void* slot_global_ptr;

typedef float slot_f32x4_t __attribute__((ext_vector_type(4)));
template <bool NARROW>
__device__ __forceinline__ f32x16_t slot_mfma(bf16x8_t a, bf16x8_t b, bf16x8_t b2, f32x16_t c) {
    if (!NARROW) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    slot_f32x4_t lo = {c[0], c[1], c[2], c[3]}, hi = {c[4], c[5], c[6], c[7]};
    lo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, lo, 0, 0, 0);
    hi = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b2, hi, 0, 0, 0);
    c[0] = lo[0]; c[1] = lo[1]; c[2] = lo[2]; c[3] = lo[3];
    c[4] = hi[0]; c[5] = hi[1]; c[6] = hi[2]; c[7] = hi[3];
    return c;
}

__device__ __forceinline__ void slot_fills(unsigned char* lds, const unsigned char* src, int wave8, int lane) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int blk = i * 8 + wave8;
        __builtin_amdgcn_global_load_lds((slot_global_ptr)(src + (size_t)blk * 1024 + lane * 16), (slot_lds_ptr)(lds + blk * 1024),
                                         16, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ void slot_end(bool fills) {
    __builtin_amdgcn_sched_barrier(0);
    if (fills) __builtin_amdgcn_s_waitcnt(0x0070);      // vmcnt(0) lgkmcnt(0)
    else __builtin_amdgcn_s_waitcnt(0xc07f);            // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
}

template <bool LDS, bool PREFETCH, bool NARROW>
__device__ __forceinline__ void slot_products(int what, int iters, unsigned char* k_lds, unsigned char* v_lds,
                                              const unsigned char* pool, float* sink) {
    const int lane = threadIdx.x & 63, wave8 = threadIdx.x >> 6, r = lane & 31, half = lane >> 5;
    const bool fills = (what & kSlotFills) != 0;
    const int k_rd = r * kSlotRowBytes;
    const int i16 = lane & 15;
    const int v_row = 4 * half + (i16 >> 2);
    const int v_col_bytes = (16 * ((lane >> 4) & 1) + 4 * (i16 & 3)) * 2;
    const int v_swz = (i16 >> 2) << 2;
    int v_rd[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        v_rd[i] = v_row * kSlotRowBytes + ((((4 * i + (v_col_bytes >> 4)) ^ v_swz) << 4) | (v_col_bytes & 15));
    const int k_swz = (half ^ (r & 15)) << 4;
    const int pattern = (what & kSlotRandom) ? 2 : 1;
    f32x16_t o_acc[4], s[4];
    bf16x8_t qf[8], pf[8];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) { o_acc[i][e] = 0.f; s[i][e] = 0.f; }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        qf[i] = probe_fragment(pattern, threadIdx.x * 16 + i);
        pf[i] = probe_fragment(pattern, threadIdx.x * 16 + 8 + i);
    }
    slot_s16x4_t vlo[2][4], vhi[2][4];
    bf16x8_t kf[2][4];
    auto v_first = [&](const unsigned char* v_blk, int b, int i) __attribute__((always_inline)) {
        const unsigned char* src = v_blk + 16 * b * kSlotRowBytes + v_rd[i];
        vlo[b][i] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((slot_lds_s16x4_ptr)src);
        vhi[b][i] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((slot_lds_s16x4_ptr)(src + 8 * kSlotRowBytes));
    };
    if (LDS && PREFETCH) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) v_first(v_lds, b, i);
    }
    for (int it = 0; it < iters; ++it) {
        if (fills)
            slot_fills((it & 1) ? k_lds + ((it + 1) & 1) * kSlotBlockBytes : v_lds + (it & 1) * kSlotBlockBytes,
                       pool + (size_t)(it & 1023) * kSlotBlockBytes, wave8, lane);
        if (!LDS) {
#pragma unroll
            for (int t2 = 0; t2 < 8; ++t2)
#pragma unroll
                for (int i = 0; i < 4; ++i) o_acc[i] = slot_mfma<NARROW>(qf[t2], pf[t2], pf[(t2 + 3) & 7], o_acc[i]);
#pragma unroll
            for (int ks = 0; ks < 8; ++ks)
#pragma unroll
                for (int j = 0; j < 4; ++j) s[j] = slot_mfma<NARROW>(pf[ks], qf[ks], qf[(ks + 3) & 7], s[j]);
        } else {
            const unsigned char* v_blk = v_lds + (it & 1) * kSlotBlockBytes;
            const unsigned char* v_nxt = v_lds + ((it + 1) & 1) * kSlotBlockBytes;
            const unsigned char* k_row = k_lds + (it & 1) * kSlotBlockBytes + k_rd;
            int swz = k_swz;
            asm volatile("" : "+v"(swz));
            auto k_read = [&](int b, int j, int ks) __attribute__((always_inline)) {
                kf[b][j] = *reinterpret_cast<const bf16x8_t*>(k_row + 32 * j * kSlotRowBytes + (swz ^ (32 * ks)));
            };
            // O^T += V^T . P^T
            if (!PREFETCH) {
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int i = 0; i < 4; ++i) v_first(v_blk, b, i);
                __builtin_amdgcn_sched_group_barrier(0x100, 16, 0);
            }
#pragma unroll
            for (int t2 = 0; t2 < 8; ++t2) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const slot_s16x4_t lo = vlo[t2 & 1][i], hi = vhi[t2 & 1][i];
                    const slot_s16x8_t both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                    o_acc[i] = slot_mfma<NARROW>(__builtin_bit_cast(bf16x8_t, both), pf[t2], pf[(t2 + 3) & 7], o_acc[i]);
                    if (t2 + 2 < 8) {
                        const unsigned char* src = v_blk + 16 * (t2 + 2) * kSlotRowBytes + v_rd[i];
                        vlo[t2 & 1][i] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((slot_lds_s16x4_ptr)src);
                        vhi[t2 & 1][i] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((slot_lds_s16x4_ptr)(src + 8 * kSlotRowBytes));
                    } else if (PREFETCH) {
                        k_read(t2 & 1, i, t2 & 1);           // the first two steps of Q.K, asked for in the tail of P.V
                    }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    if (t2 + 2 < 8) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                    else if (PREFETCH) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                }
            }
            // S^T = K . Q^T
            if (!PREFETCH) {
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int j = 0; j < 4; ++j) k_read(b, j, b);
                __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
            }
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    s[j] = slot_mfma<NARROW>(kf[ks & 1][j], qf[ks], qf[(ks + 3) & 7], s[j]);
                    if (ks + 2 < 8) k_read(ks & 1, j, ks + 2);
                    else if (PREFETCH) v_first(v_nxt, ks & 1, j);   // the next slot's first two steps of P.V
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    if (ks + 2 < 8) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    else if (PREFETCH) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                }
            }
        }
        slot_end(fills);
    }
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) t += o_acc[i][e] + s[i][e];
    if (LDS && PREFETCH) t += (float)vlo[0][0][0] + (float)vhi[1][3][1];
    sink[blockIdx.x * 512 + threadIdx.x] = t;
}

__device__ __forceinline__ void slot_softmax(int what, int iters, unsigned char* k_lds, unsigned char* v_lds,
                                             const unsigned char* pool, float* sink) {
    const int lane = threadIdx.x & 63, wave8 = threadIdx.x >> 6;
    const bool fills = (what & kSlotFills) != 0;
    float s[64];
#pragma unroll
    for (int e = 0; e < 64; ++e) s[e] = (float)(probe_hash(threadIdx.x * 64 + e) & 0xffff) * (1.0f / 4096.f);
    float m_i = -1e30f, l_i = 0.f;
    unsigned packed = 0;
    for (int it = 0; it < iters; ++it) {
        if (fills)
            slot_fills((it & 1) ? k_lds + ((it + 1) & 1) * kSlotBlockBytes : v_lds + (it & 1) * kSlotBlockBytes,
                       pool + (size_t)(it & 1023) * kSlotBlockBytes, wave8, lane);
#pragma unroll
        for (int e = 0; e < 64; ++e) asm volatile("" : "+v"(s[e]));      // new scores every slot, as far as the compiler knows
        float mx = -1e30f;
#pragma unroll
        for (int e = 0; e < 64; ++e) mx = fmaxf(mx, s[e]);
        const float m_new = fmaxf(m_i, mx * 0.088f);
        const float alpha = __builtin_amdgcn_exp2f(m_i - m_new);
        float row = 0.f;
#pragma unroll
        for (int e = 0; e < 64; e += 2) {
            const float p0 = __builtin_amdgcn_exp2f(s[e] * 0.088f - m_new);
            const float p1 = __builtin_amdgcn_exp2f(s[e + 1] * 0.088f - m_new);
            row += p0;
            row += p1;
            typedef __bf16 bf16x2_slot_t __attribute__((ext_vector_type(2)));
            const bf16x2_slot_t pk = {(__bf16)p0, (__bf16)p1};
            unsigned u = __builtin_bit_cast(unsigned, pk);
            asm volatile("" : "+v"(u));
            packed ^= u;
        }
        l_i = l_i * alpha + row;
        m_i = m_new;
        slot_end(fills);
    }
    sink[blockIdx.x * 512 + threadIdx.x] = l_i + m_i + (float)packed;
}

template <bool LDS, bool PREFETCH, bool NARROW>
__global__ void __launch_bounds__(512, 1) attn_slot_kernel(int what, int iters, const unsigned char* pool, float* sink,
                                                           long long* cycles) {
    __shared__ __attribute__((aligned(1024))) unsigned char k_lds[2 * kSlotBlockBytes];
    __shared__ __attribute__((aligned(1024))) unsigned char v_lds[2 * kSlotBlockBytes];
    for (int i = threadIdx.x; i < 2 * kSlotBlockBytes / 4; i += 512) {
        unsigned a = 0x3c003c00u, b = 0x3c003c00u;
        if (what & kSlotRandom) {
            const bf16x8_t f = probe_fragment(2, blockIdx.x * 65536 + i);
            const u32x4_probe_t w = __builtin_bit_cast(u32x4_probe_t, f);
            a = w[0];
            b = w[1];
        }
        reinterpret_cast<unsigned*>(k_lds)[i] = a;
        reinterpret_cast<unsigned*>(v_lds)[i] = b;
    }
    __syncthreads();
    const int wave8 = threadIdx.x >> 6;
    const unsigned char* mine = (what & kSlotPrivate) ? pool + (size_t)blockIdx.x * 65536 : pool;
    const long long t0 = clock64();
    if (wave8 < 4) {
        if (what & kSlotProducts) slot_products<LDS, PREFETCH, NARROW>(what, iters, k_lds, v_lds, mine, sink);
        else for (int it = 0; it < iters; ++it) __builtin_amdgcn_s_barrier();
    } else {
        if (what & kSlotSoftmax) slot_softmax(what, iters, k_lds, v_lds, mine, sink);
        else for (int it = 0; it < iters; ++it) __builtin_amdgcn_s_barrier();
    }
    const long long t1 = clock64();
    if (blockIdx.x == 0 && (threadIdx.x & 255) == 0) cycles[wave8 >> 2] = t1 - t0;
}

// The same streams read the way the reduce's skewed walk reads them: a workgroup takes eight consecutive blocks of
// 4 KB per stream and in step t reads block t - i of stream i, the next step's loads issued before this step's are used.
template <int STREAMS>
__global__ void __launch_bounds__(kStreamThreads)
read_streams_skewed_kernel(const u32x4_probe_t* __restrict__ base, int64_t stride_vecs, int64_t stream_vecs,
                           u32x4_probe_t* __restrict__ sink) {
    constexpr int kBlocks = 8;
    constexpr int64_t kSuper = (int64_t)kStreamThreads * kBlocks;
    constexpr int kSteps = kBlocks + STREAMS - 1;
    u32x4_probe_t mix = {0u, 0u, 0u, 0u};
    for (int64_t g0 = (int64_t)blockIdx.x * kSuper; g0 + kSuper <= stream_vecs; g0 += (int64_t)gridDim.x * kSuper) {
        u32x4_probe_t even[STREAMS], odd[STREAMS];
        auto issue = [&](const int t, u32x4_probe_t (&dst)[STREAMS]) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < STREAMS; ++i) {
                const int b = t - i;
                if (b >= 0 && b < kBlocks)
                    dst[i] = __builtin_nontemporal_load(base + (int64_t)i * stride_vecs + g0 + b * kStreamThreads + threadIdx.x);
            }
        };
        auto take = [&](const int t, const u32x4_probe_t (&src)[STREAMS]) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < STREAMS; ++i) {
                const int b = t - i;
                if (b >= 0 && b < kBlocks) mix ^= src[i];
            }
        };
        issue(0, even);
#pragma unroll
        for (int t = 0; t < kSteps; ++t) {
            if (t + 1 < kSteps) {
                if (t & 1) issue(t + 1, even);
                else issue(t + 1, odd);
            }
            if (t & 1) take(t, odd);
            else take(t, even);
        }
    }
    if ((mix.x ^ mix.y ^ mix.z ^ mix.w) == 0x9e3779b9u) sink[blockIdx.x] = mix;
}

}  // namespace syn

extern "C" int syn_probe_read_streams(const void* base, int64_t stream_bytes, int64_t stride_bytes, int32_t streams,
                                      int32_t workgroups, void* sink, syn_stream_t stream) {
    using namespace syn;
    if (base == nullptr || sink == nullptr || workgroups <= 0) return SYN_EINVAL;
    if (stream_bytes <= 0 || stream_bytes % (16 * kStreamThreads * kStreamVecs)) return SYN_EINVAL;
    if (streams != 1 && streams != 8) return SYN_EINVAL;
    if (stride_bytes < 0 || stride_bytes % 16 || !aligned16(base) || !aligned16(sink)) return SYN_EALIGN;
    const u32x4_probe_t* b = reinterpret_cast<const u32x4_probe_t*>(base);
    u32x4_probe_t* k = reinterpret_cast<u32x4_probe_t*>(sink);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (streams == 1)
        hipLaunchKernelGGL(read_streams_kernel<1>, dim3(workgroups), dim3(kStreamThreads), 0, s, b, stride_bytes / 16,
                           stream_bytes / 16, k);
    else
        hipLaunchKernelGGL(read_streams_kernel<8>, dim3(workgroups), dim3(kStreamThreads), 0, s, b, stride_bytes / 16,
                           stream_bytes / 16, k);
    return (int)hipGetLastError();
}

extern "C" int syn_probe_read_streams_skewed(const void* base, int64_t stream_bytes, int64_t stride_bytes, int32_t workgroups,
                                             void* sink, syn_stream_t stream) {
    using namespace syn;
    if (base == nullptr || sink == nullptr || workgroups <= 0) return SYN_EINVAL;
    if (stream_bytes <= 0 || stream_bytes % (16 * kStreamThreads * 8)) return SYN_EINVAL;
    if (stride_bytes < 0 || stride_bytes % 16 || !aligned16(base) || !aligned16(sink)) return SYN_EALIGN;
    hipLaunchKernelGGL(read_streams_skewed_kernel<8>, dim3(workgroups), dim3(kStreamThreads), 0,
                       reinterpret_cast<hipStream_t>(stream), reinterpret_cast<const u32x4_probe_t*>(base), stride_bytes / 16,
                       stream_bytes / 16, reinterpret_cast<u32x4_probe_t*>(sink));
    return (int)hipGetLastError();
}

extern "C" int syn_probe_mfma_rate(float* sink, int32_t workgroups, int32_t iters, int32_t pattern,
                                   syn_stream_t stream) {
    using namespace syn;
    // bits 0-1: operands; 2: the MFMA; 4-5: the order, of the 16x16x32 form
    const int order = pattern >> 4;
    if (sink == nullptr || workgroups <= 0 || iters <= 0 || pattern < 0 || (pattern & 3) > 2 || (pattern & 8) || order > 3)
        return SYN_EINVAL;
    if (order != 0 && !(pattern & 4)) return SYN_EINVAL;
    auto* const kernel = !(pattern & 4)              ? mfma_rate_kernel
                         : order == kOrderPairs      ? mfma16_rate_kernel<kOrderPairs>
                         : order == kOrderRows       ? mfma16_rate_kernel<kOrderRows>
                         : order == kOrderToAndFro   ? mfma16_rate_kernel<kOrderToAndFro>
                                                     : mfma16_rate_kernel<kOrderDiagonal>;
    hipLaunchKernelGGL(kernel, dim3(workgroups), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), sink, iters, pattern & 3);
    return (int)hipGetLastError();
}

extern "C" int syn_probe_attn_slot(const void* pool, int64_t pool_bytes, int32_t workgroups, int32_t iters, int32_t what,
                                   float* sink, int64_t* cycles, syn_stream_t stream) {
    using namespace syn;
    if (pool == nullptr || sink == nullptr || cycles == nullptr || workgroups <= 0 || iters <= 0) return SYN_EINVAL;
    if (what <= 0 || what >= 256 || !(what & (kSlotProducts | kSlotSoftmax))) return SYN_EINVAL;
    if ((what & kSlotNarrow) && !(what & kSlotProducts)) return SYN_EINVAL;
    if ((what & kSlotPrefetch) && !(what & kSlotLds)) return SYN_EINVAL;
    // a workgroup's fills read 32 KB pieces at pool (+ 64 KB * workgroup with kSlotPrivate) + 32 KB * (slot % 1024)
    if (pool_bytes < (int64_t)workgroups * 65536 + 1024 * (int64_t)kSlotBlockBytes) return SYN_EINVAL;
    if (!aligned16(pool)) return SYN_EALIGN;
    const unsigned char* g = reinterpret_cast<const unsigned char*>(pool);
    long long* c = reinterpret_cast<long long*>(cycles);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const dim3 grid(workgroups), block(512);
    const bool narrow = (what & kSlotNarrow) != 0;
    if (!(what & kSlotLds)) {
        if (narrow) hipLaunchKernelGGL((attn_slot_kernel<false, false, true>), grid, block, 0, s, what, iters, g, sink, c);
        else hipLaunchKernelGGL((attn_slot_kernel<false, false, false>), grid, block, 0, s, what, iters, g, sink, c);
    } else if (what & kSlotPrefetch) {
        if (narrow) hipLaunchKernelGGL((attn_slot_kernel<true, true, true>), grid, block, 0, s, what, iters, g, sink, c);
        else hipLaunchKernelGGL((attn_slot_kernel<true, true, false>), grid, block, 0, s, what, iters, g, sink, c);
    } else {
        if (narrow) hipLaunchKernelGGL((attn_slot_kernel<true, false, true>), grid, block, 0, s, what, iters, g, sink, c);
        else hipLaunchKernelGGL((attn_slot_kernel<true, false, false>), grid, block, 0, s, what, iters, g, sink, c);
    }
    return (int)hipGetLastError();
}
