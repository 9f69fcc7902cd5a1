// Scaled-dot-product attention for head_dim 64 (fp16 in and out, fp32 softmax
// and accumulation), non-causal, no mask: the decoder attention of the H3 VAE
// that the reference hands to the model's `perform_attention` (flash attention
// on NVIDIA) between the fused QK-RMSNorm-RoPE and the INT8 attention-out
// linear (opt/decoder_fused_qk_rope.py:66-74, `FusedQKAttention.forward`).
//
//   O[q, :] = sum_k softmax_k(scale * Q[q, :] . K[k, :]) V[k, :]
//
// q, k, v, o are [batch, tokens, heads, 64] with arbitrary token and head
// strides (in elements; the 64 dims contiguous), so v can be the strided
// slice of the QKV projection and q, k the QK-RoPE outputs, with no copies.
//
// One workgroup = 8 waves = 512 queries of one (batch, head); each wave owns
// two sets of 32 queries (one set, or 4 waves, where that fills the chip better,
// see plan_attention).  Keys and values stream in blocks of 64 through LDS:
//
//   S = K . Q^T   v_mfma_f32_32x32x16_f16, A = K rows from LDS, B = the wave's
//                 Q fragments (registers, loaded once).  In the 32 x 32 result
//                 layout lane l holds query l % 32 and keys 8g + 4(l / 32) + e
//                 (g, e = 0..3) of each 32-key half, so a query's 64 keys sit
//                 in lanes l and l ^ 32 (32 each): the row max and sum are
//                 in-lane reductions plus one exchange.
//   online softmax in fp32 (exp2 with the scale folded into log2 e) against a
//                 lazy reference maximum that moves only when a weight would
//                 exceed 2^8; the row sums add the fp16-rounded weights that the
//                 P.V product uses
//   O^T += V^T . P^T   A = V^T rows from LDS (V is written transposed), B = P
//                 in fp16: one v_permlane32_swap per dword pair turns the S
//                 layout into the MFMA's 8 consecutive keys per lane.
//
// LDS: three slots of K [64 keys][64 dims] and V^T [64 dims][64 keys] fp16,
// 128-byte rows whose 16-byte chunks are XOR-swizzled by (row >> 1) & 7, so the
// 16-lane fragment reads hit 16 distinct 4-bank groups.  K and V of block j + 2
// are loaded into registers while block j is computed and stored into their
// slot after the next barrier; waves 4-7 run one phase behind waves 0-3 (see
// the main loop).
#include "h3v_common.hpp"
#include "h3v_abi.hpp"

namespace h3v {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kD = 64;        // head dim
constexpr int kBK = 64;       // keys per block
constexpr int kThreads = 256;   // the K / V loading threads (waves 0-3 of a workgroup)
constexpr float kLazy = 8.0f;   // log2 margin of the lazy softmax maximum (weights stay <= 2^kLazy)
constexpr int kSlots = 3;       // K / V^T blocks resident in LDS (block j in slot j % 3)

struct AttnParams {
    const uint16_t* q;
    const uint16_t* k;
    const uint16_t* v;
    uint16_t* o;
    int64_t q_ts, q_hs, k_ts, k_hs, v_ts, v_hs, o_ts, o_hs;
    int tokens;
    float c;   // scale * log2(e)
    int q_first;   // first query of the launch
    // key splits: split sp of a batch item sees key blocks sp * split_blocks ... (splits = 1: all of them)
    int splits, split_blocks;
    float* part;   // PART: [splits][batch * heads][tokens - q_first] rows of 64 unnormalised outputs
    float* ml;     // PART: as many (reference maximum, weight sum) pairs
};

__device__ __forceinline__ int swz(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }

__device__ __forceinline__ float wave_pair_max(float v) { return __builtin_fmaxf(v, __shfl_xor(v, 32, 64)); }

// two fp32 -> packed fp16 (round to nearest even), one v_cvt_pk_f16_f32
__device__ __forceinline__ uint32_t pack_f16x2(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, f16x2));
}

// QS sets of 32 queries per wave, NW waves (8 or 4; 32 * NW * QS queries per workgroup); every K and V^T
// fragment read from LDS feeds the MFMAs of all QS sets (two sets: 233 VGPRs, 2 waves per SIMD; one: 150, 3
// waves).  Waves 0-3 move each K / V block into LDS for all 8 (half the per-query load and transpose work of
// 4-wave workgroups).  Every query goes through the same operations in the same order whatever QS and NW are, but
// for the blocks that move a reference maximum, which the queries of a wave do together.
// PART: one split of the keys, its unnormalised outputs and (m_ref, sum) pairs to p.part / p.ml (fp32).
template <int QS, int NW, bool PART>
__global__ __launch_bounds__(64 * NW) void fmha_d64(AttnParams p) {
    constexpr int BQ = 32 * NW * QS;
    constexpr int KV = kBK * kD;                                      // elements of one K or V^T block
    __shared__ __attribute__((aligned(16))) uint16_t ks[kSlots * KV];   // [slot][key][dim]
    __shared__ __attribute__((aligned(16))) uint16_t vt[kSlots * KV];   // [slot][dim][key]

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform (scalar)
    const int h = blockIdx.y, b = PART ? blockIdx.z / p.splits : blockIdx.z;
    const int n = p.tokens;
    const int64_t row0 = (int64_t)b * n;                 // first token row of this batch item
    // the wave's first query; only the one-set workgroups run the queries past others
    const int q0 = (QS == 1 ? p.q_first : 0) + blockIdx.x * BQ + wave * 32 * QS;
    const int hi = lane >> 5;                           // which 8 of a 16-wide k chunk this lane holds
    const bool wave_active = q0 < n;                    // wave-uniform

    // the wave's Q fragments: query q0 + 32 qs + lane % 32, dims 16 kc + 8 hi .. + 7
    half8 qf[QS][4];
#pragma unroll
    for (int qs = 0; qs < QS; ++qs) {
        const int qi = q0 + 32 * qs + (lane & 31);
        const int qr = qi < n ? qi : n - 1;
        const uint16_t* src = p.q + (row0 + qr) * p.q_ts + h * p.q_hs + 8 * hi;
#pragma unroll
        for (int kc = 0; kc < 4; ++kc) qf[qs][kc] = *reinterpret_cast<const half8*>(src + 16 * kc);
    }

    // cooperative K / V block loads.  K: 64 keys x 8 chunks of 8 dims = 512 chunks, two per thread,
    // consecutive threads walking a key row.  V: each thread reads a 4-key x 4-dim block (four
    // 8-byte loads; 16 consecutive threads cover one 128-byte key row) and transposes it in
    // registers, so the V^T rows go to LDS as four 8-byte stores of 4 consecutive keys each.
    u32x4 kreg[2];
    uint32_t vreg[4][2];                                  // [key of the 4][dims 0-1, 2-3]
    const int vdg = tid & 15, vkg = tid >> 4;             // dims 4 vdg .. +3, keys 4 vkg .. +3
    // Per-thread source rows of block 0; a full block adds the uniform kb0 * stride (scalar),
    // only the last, partial block clamps rows past the end to the last token.
    const uint16_t* kbase[2];
    const uint16_t* vbase[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int c = tid + kThreads * i;
        kbase[i] = p.k + (row0 + (c >> 3)) * p.k_ts + h * p.k_hs + 8 * (c & 7);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) vbase[i] = p.v + (row0 + 4 * vkg + i) * p.v_ts + h * p.v_hs + 4 * vdg;
    auto load_block = [&](int kb0) {
        if (kb0 + kBK <= n) {
            const int64_t ko = (int64_t)kb0 * p.k_ts, vo = (int64_t)kb0 * p.v_ts;
#pragma unroll
            for (int i = 0; i < 2; ++i) kreg[i] = *reinterpret_cast<const u32x4*>(kbase[i] + ko);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint2 w = *reinterpret_cast<const uint2*>(vbase[i] + vo);
                vreg[i][0] = w.x;
                vreg[i][1] = w.y;
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int c = tid + kThreads * i;
            const int key = c >> 3, dch = c & 7;
            const int kr = kb0 + key < n ? kb0 + key : n - 1;
            kreg[i] = *reinterpret_cast<const u32x4*>(p.k + (row0 + kr) * p.k_ts + h * p.k_hs + 8 * dch);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int key = 4 * vkg + i;
            const int vr = kb0 + key < n ? kb0 + key : n - 1;
            const uint2 w = *reinterpret_cast<const uint2*>(p.v + (row0 + vr) * p.v_ts + h * p.v_hs + 4 * vdg);
            vreg[i][0] = w.x;
            vreg[i][1] = w.y;
        }
    };
    auto store_block = [&](int slot) {
        uint16_t* const kd = ks + slot * KV;
        uint16_t* const vd = vt + slot * KV;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int c = tid + kThreads * i;
            const int key = c >> 3, dch = c & 7;
            *reinterpret_cast<u32x4*>(kd + key * kD + 8 * swz(key, dch)) = kreg[i];
        }
        // dim j of the 4: keys 0-1 from the low (j even) or high (j odd) halves of vreg[0..1][j >> 1],
        // keys 2-3 likewise from vreg[2..3]; v_perm_b32 picks the two halves into one dword
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
            const uint32_t lo = __builtin_amdgcn_perm(vreg[1][j >> 1], vreg[0][j >> 1], sel);
            const uint32_t hi = __builtin_amdgcn_perm(vreg[3][j >> 1], vreg[2][j >> 1], sel);
            const int d = 4 * vdg + j;
            *reinterpret_cast<uint2*>(vd + d * kBK + 8 * swz(d, vkg >> 1) + 4 * (vkg & 1)) = make_uint2(lo, hi);
        }
    };

    f32x16 oacc[QS][2];
    float m_ref[QS], mc[QS], l_run[QS];
#pragma unroll
    for (int qs = 0; qs < QS; ++qs) {
        oacc[qs][0] = f32x16{};
        oacc[qs][1] = f32x16{};
        m_ref[qs] = -__builtin_inff();
        mc[qs] = PART ? 0.0f : -__builtin_inff();
        l_run[qs] = 0.0f;
    }
    const float thr = kLazy / p.c;   // raw-score margin of the lazy maximum

    const int sp = PART ? (int)blockIdx.z % p.splits : 0;
    const int j0 = sp * p.split_blocks;                   // this workgroup's key blocks: j0 .. nblk - 1
    const int nall = (n + kBK - 1) / kBK;
    const int nblk = PART && j0 + p.split_blocks < nall ? j0 + p.split_blocks : nall;
    const bool loader = tid < kThreads;                   // waves 0-3 (wave-uniform)

    // S = K . Q^T for the 64 keys of block j (two 32-key halves), each K fragment used by every set;
    // keys past the end (last block only) are -inf
    auto scores = [&](int j, int slot, f32x16 (&s)[QS][2]) {
        const int kb0 = j * kBK;
        const uint16_t* const kb = ks + slot * KV;
#pragma unroll
        for (int kh = 0; kh < 2; ++kh) {
#pragma unroll
            for (int qs = 0; qs < QS; ++qs) s[qs][kh] = f32x16{};
            const int row = 32 * kh + (lane & 31);
#pragma unroll
            for (int kc = 0; kc < 4; ++kc) {
                const half8 a = *reinterpret_cast<const half8*>(kb + row * kD + 8 * swz(row, 2 * kc + hi));
#pragma unroll
                for (int qs = 0; qs < QS; ++qs)
                    s[qs][kh] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qf[qs][kc], s[qs][kh], 0, 0, 0);
            }
        }
        if (kb0 + kBK > n) {
#pragma unroll
            for (int qs = 0; qs < QS; ++qs)
#pragma unroll
                for (int kh = 0; kh < 2; ++kh)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int key = kb0 + 32 * kh + 8 * (r >> 2) + 4 * hi + (r & 3);
                        if (key >= n) s[qs][kh][r] = -__builtin_inff();
                    }
        }
    };
    // online softmax per set in raw-score units (the exponent folds in scale * log2 e), with a lazy
    // reference maximum: the weights are exp2(s * c - m_ref * c), and m_ref moves (rescaling O and l by
    // exp2((m_old - m_ref) * c)) only when a score of the block exceeds it by more than kLazy / c, i.e.
    // when a weight would exceed 2^kLazy.  Every weight stays in [0, 256], where fp16 keeps the same
    // relative precision, and after the first block the 64 rescale multiplies almost never run (with
    // the exact running maximum some lane's maximum moves in nearly every block).  P in fp16.
    auto softmax = [&](const f32x16 (&s)[QS][2], uint32_t (&pk)[QS][2][8]) {
        bool up = false;
        float mblk[QS];
#pragma unroll
        for (int qs = 0; qs < QS; ++qs) {
            float mloc = s[qs][0][0];
#pragma unroll
            for (int kh = 0; kh < 2; ++kh)
#pragma unroll
                for (int r = 0; r < 16; ++r) mloc = __builtin_fmaxf(mloc, s[qs][kh][r]);
            mblk[qs] = wave_pair_max(mloc);
            up |= mblk[qs] > m_ref[qs] + thr;   // m_ref = -inf before the first block: true there
        }
        if (__ballot(up)) {
#pragma unroll
            for (int qs = 0; qs < QS; ++qs) {
                const float m_new = __builtin_fmaxf(m_ref[qs], mblk[qs]);
                float alpha = __builtin_amdgcn_exp2f((m_ref[qs] - m_new) * p.c);   // 0 from -inf, 1 if unmoved
                m_ref[qs] = m_new;
                mc[qs] = m_new * p.c;
                if constexpr (PART) {
                    // a split whose scores are all -inf so far has weights of 0 (another split has the others)
                    if (m_new == -__builtin_inff()) {
                        alpha = 1.0f;
                        mc[qs] = 0.0f;
                    }
                }
                l_run[qs] *= alpha;
#pragma unroll
                for (int db = 0; db < 2; ++db)
#pragma unroll
                    for (int r = 0; r < 16; ++r) oacc[qs][db][r] *= alpha;
            }
        }
#pragma unroll
        for (int qs = 0; qs < QS; ++qs) {
            float lsum = 0.0f;
#pragma unroll
            for (int kh = 0; kh < 2; ++kh)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    float e4[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        e4[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[qs][kh][4 * g + e], p.c, -mc[qs]));
                    pk[qs][kh][2 * g] = pack_f16x2(e4[0], e4[1]);
                    pk[qs][kh][2 * g + 1] = pack_f16x2(e4[2], e4[3]);
                    // the row sum adds the fp16 weights the P.V product uses, two per v_dot2_f32_f16
                    const f16x2 one = {(_Float16)1.0f, (_Float16)1.0f};
                    lsum = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, pk[qs][kh][2 * g]), one, lsum, false);
                    lsum = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, pk[qs][kh][2 * g + 1]), one, lsum, false);
                }
            l_run[qs] += lsum;
        }
    };
    // O^T += V^T . P^T over four 16-key chunks, each V^T fragment used by every set.  (With both wave
    // groups in one phase a raised issue priority for these MFMAs had paid, 153.7 -> 151.5 us on the H3
    // call; with the groups a phase apart it costs: 146.8 us without it against 149.5 us.)
    auto pv = [&](int slot, const uint32_t (&pk)[QS][2][8]) {
        const uint16_t* const vb = vt + slot * KV;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int kh = c >> 1, g0 = 2 * (c & 1);
            // lane < 32 needs keys 16c + 0..7 (its own group g0 + the partner's), lane >= 32
            // keys 16c + 8..15 (the partner's group g0 + 1 + its own)
            half8 bop[QS];
#pragma unroll
            for (int qs = 0; qs < QS; ++qs) {
                const auto x0 = __builtin_amdgcn_permlane32_swap(pk[qs][kh][2 * g0], pk[qs][kh][2 * g0 + 2], false, false);
                const auto x1 = __builtin_amdgcn_permlane32_swap(pk[qs][kh][2 * g0 + 1], pk[qs][kh][2 * g0 + 3], false,
                                                                 false);
                const u32x4 bw = {x0[0], x1[0], x0[1], x1[1]};
                bop[qs] = __builtin_bit_cast(half8, bw);
            }
#pragma unroll
            for (int db = 0; db < 2; ++db) {
                const int row = 32 * db + (lane & 31);
                const half8 a = *reinterpret_cast<const half8*>(vb + row * kBK + 8 * swz(row, 2 * c + hi));
#pragma unroll
                for (int qs = 0; qs < QS; ++qs)
                    oacc[qs][db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, bop[qs], oacc[qs][db], 0, 0, 0);
            }
        }
    };

    // One barrier per block, three LDS slots.  Waves 0-3 (the loaders) run block j as scores, softmax,
    // P.V after barrier j; waves 4-7 run the P.V of block j - 1 and then the scores and softmax of block
    // j, carrying the packed weights P over the barrier.  On each SIMD one wave's softmax VALU work then
    // runs beside its partner's MFMAs for two of the three phases instead of both waves running the
    // same phase; every query sees the same operations in the same order.  After barrier j the loaders
    // store block j + 1 into slot (j + 1) % 3, which last held block j - 2: its readers finished before
    // barrier j (waves 4-7 read it in their iteration j - 1); block j + 1 is read only after barrier
    // j + 1.  The two groups run separate loops with one barrier per iteration each.
    // The Q fragment loads complete here, once: otherwise the wait counters merged over the loop's back
    // edge keep them pending, and the first score MFMAs of every block wait for that block's K / V loads.
    __builtin_amdgcn_s_waitcnt(0);
    uint32_t pk[QS][2][8];                                // [set][half][g * 2 + dword]
    if (loader) {
        load_block(j0 * kBK);
        store_block(0);
        if (j0 + 1 < nblk) load_block((j0 + 1) * kBK);
        int slot = 0;                                     // slot of block j
        for (int j = j0; j < nblk; ++j) {
            __syncthreads();                              // block j stored; blocks before j - 1 no longer read
            const int nslot = slot == kSlots - 1 ? 0 : slot + 1;
            if (j + 1 < nblk) {
                store_block(nslot);
                if (j + 2 < nblk) load_block((j + 2) * kBK);   // block j + 2 in flight during this one
            }
            // a wave whose 32 queries all lie past the end (the last workgroup of a head) only helps
            // with the shared K / V loads and barriers
            if (wave_active) {
                f32x16 s[QS][2];
                scores(j, slot, s);
                softmax(s, pk);
                pv(slot, pk);
            }
            slot = nslot;
        }
    } else {
        int slot = 0, pslot = 0;                          // slots of blocks j and j - 1
        for (int j = j0; j < nblk; ++j) {
            __syncthreads();
            if (wave_active) {
                if (j > j0) pv(pslot, pk);
                f32x16 s[QS][2];
                scores(j, slot, s);
                softmax(s, pk);
            }
            pslot = slot;
            slot = slot == kSlots - 1 ? 0 : slot + 1;
        }
        if (wave_active) pv(pslot, pk);                   // the last block (no store follows it)
    }

    // normalise and store: lane l holds query q0 + 32 qs + l % 32, dims 32 db + 8 g + 4 hi + e
#pragma unroll
    for (int qs = 0; qs < QS; ++qs) {
        const int qi = q0 + 32 * qs + (lane & 31);
        const float l_tot = l_run[qs] + __shfl_xor(l_run[qs], 32, 64);
        if constexpr (PART) {
            if (qi < n) {
                const int64_t row = ((int64_t)(sp * (gridDim.z / p.splits) + b) * gridDim.y + h) * (n - p.q_first) +
                                    (qi - p.q_first);
                float* dst = p.part + row * kD + 4 * hi;
#pragma unroll
                for (int db = 0; db < 2; ++db)
#pragma unroll
                    for (int g = 0; g < 4; ++g)
                        *reinterpret_cast<float4*>(dst + 32 * db + 8 * g) =
                            make_float4(oacc[qs][db][4 * g], oacc[qs][db][4 * g + 1], oacc[qs][db][4 * g + 2],
                                        oacc[qs][db][4 * g + 3]);
                if (hi == 0) *reinterpret_cast<float2*>(p.ml + 2 * row) = make_float2(m_ref[qs], l_tot);
            }
            continue;
        }
        const float inv = 1.0f / l_tot;
        if (qi < n) {
            uint16_t* dst = p.o + (row0 + qi) * p.o_ts + h * p.o_hs + 4 * hi;
#pragma unroll
            for (int db = 0; db < 2; ++db)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    u16x4 v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = f2h(oacc[qs][db][4 * g + e] * inv);
                    *reinterpret_cast<u16x4*>(dst + 32 * db + 8 * g) = v;
                }
        }
    }
}

// Merge of the key splits: per query the splits' outputs and sums rescaled to their largest reference maximum,
// added in split order, normalised.  16 threads per query, 4 dims each.
__global__ __launch_bounds__(256) void fmha_merge(AttnParams p, int heads, int64_t rows) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t row = i >> 4;
    if (row >= rows) return;
    const int d = 4 * (int)(i & 15);
    float m = -__builtin_inff();
    for (int sp = 0; sp < p.splits; ++sp) m = __builtin_fmaxf(m, p.ml[2 * (sp * rows + row)]);
    float l = 0.0f, o[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int sp = 0; sp < p.splits; ++sp) {
        const float2 ml = *reinterpret_cast<const float2*>(p.ml + 2 * (sp * rows + row));
        const float4 v = *reinterpret_cast<const float4*>(p.part + (sp * rows + row) * kD + d);
        const float w = ml.x == m ? 1.0f : __builtin_amdgcn_exp2f((ml.x - m) * p.c);
        l += w * ml.y;
        o[0] += w * v.x; o[1] += w * v.y; o[2] += w * v.z; o[3] += w * v.w;
    }
    const float inv = 1.0f / l;
    const int rest = p.tokens - p.q_first;
    const int64_t bh = row / rest;
    const int64_t t = (bh / heads) * p.tokens + p.q_first + row % rest;
    u16x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = f2h(o[e] * inv);
    *reinterpret_cast<u16x4*>(p.o + t * p.o_ts + (bh % heads) * p.o_hs + d) = y;
}

// Launches of one attention call: queries [0, head) as the workgroup shape `shape`, then the rest as 256-query
// workgroups (one set per wave), their keys split `splits` ways.
enum class AttnShape { Q512, Q256, Q256x4, Q128 };   // 8 waves x 2 sets, 8 x 1, 4 x 2, 4 x 1
struct AttnPlan {
    AttnShape shape;
    int64_t head;       // a multiple of 512, or tokens
    int splits, split_blocks;
};

// A CU holds one 8-wave workgroup of two sets, so the count of 512-query workgroups t against the 256 CUs
// decides (us for 512 / 256 / 256 on 4 waves / 128 queries; batch x tokens x 32 heads):
//   t <= 64          128 queries            1 x 453: 22.9 / 15.3 / 17.3 / 12.3, 1 x 1013: 38.1 / 26.0 / 29.9 / 22.2
//   t <= 128         256 queries            1 x 1797: 63.8 / 46.9 / 51.4 / 50.9, 4 x 453: 24.5 / 17.6 / 20.5 / 21.2
//   t <= 256         512 queries            2 x 1797: 75.0 / 87.9 / 85.2 / 92.7
// Beyond one round, workgroups of 512 for the whole rounds; the queries past them, when they are at most 128
// workgroups of 256 queries and the full rounds are nearly full, run with their keys split so that they fill the
// chip too (1 x 8405: 825.6 -> 651.7; 1 x 4100: 277.3 -> 179.1; error against 64 bits unchanged, 2.96e-4).
// Otherwise 4-wave workgroups, two of which share a CU, where the last round is at most half full, so that its
// workgroups of 256 queries find a CU each, in a call of under four rounds (or of rows so short that the rounds stay
// together): 512 against 256 on 4 waves, 3 x 1797 135.7 / 125.7, 1 x 6144 412.7 / 388.3, 1 x 10240 1046.5 / 1027.0,
// 1 x 14336 1992.9 / 1981.4, 33 x 453 125.2 / 114.2.  With the last round 5/8 full a CU gets two of them
// (1 x 6200 412.3 / 470.0, 1 x 10400 1063.4 / 1198.6), in more rounds their ends drift apart (2 x 11205 2320 / 2443,
// 13 x 1797 498.5 / 515.1), and beside another stream's call their smaller share of each key block counts: decoding
// with 3 x 1797 or 2 x 2805 tokens on two tile streams took 2% longer with them.
AttnPlan plan_attention(int64_t batch, int64_t tokens, int64_t heads, bool may_split, bool on_its_own) {
    constexpr int64_t kCUs = 256;
    const int64_t bh = batch * heads, nblk = (tokens + kBK - 1) / kBK;
    const int64_t t = (tokens + 511) / 512 * bh;
    AttnPlan plan = {AttnShape::Q512, tokens, 1, (int)nblk};
    if (t <= 64) plan.shape = AttnShape::Q128;
    else if (t <= 128) plan.shape = AttnShape::Q256;
    if (t <= kCUs || t % kCUs == 0) return plan;
    const int64_t rounds = t / kCUs, full = rounds * kCUs / bh;   // 512-query blocks per head in whole rounds
    const int64_t rest = tokens - 512 * full, w = (rest + 255) / 256 * bh;
    if (full > 0 && 16 * full * bh >= 15 * rounds * kCUs && w <= 128) {
        // split sizes of at least 4 key blocks (tokens > 512 here); they are rounded up, so the last split may be
        // shorter, down to one block
        int64_t splits = may_split ? kCUs / w : 1;
        splits = splits < nblk / 4 ? splits : nblk / 4;
        splits = splits < 1 ? 1 : (splits > 16 ? 16 : splits);
        plan.head = 512 * full;
        plan.split_blocks = (int)((nblk + splits - 1) / splits);
        plan.splits = (int)((nblk + plan.split_blocks - 1) / plan.split_blocks);
        return plan;
    }
    if (on_its_own && 2 * (t - rounds * kCUs) <= kCUs && (rounds < 4 || tokens <= 1024)) plan.shape = AttnShape::Q256x4;
    return plan;
}

int64_t attention_ws_floats(const AttnPlan& plan, int64_t batch, int64_t tokens, int64_t heads) {
    return plan.splits > 1 ? plan.splits * batch * heads * (tokens - plan.head) * (kD + 2) : 0;
}

template <int QS, int NW, bool PART>
void launch_fmha(const AttnParams& p, int64_t queries, int64_t heads, int64_t batch, hipStream_t stream) {
    constexpr int64_t BQ = 32 * NW * QS;
    const dim3 grid((unsigned)((queries + BQ - 1) / BQ), (unsigned)heads, (unsigned)(batch * p.splits));
    hipLaunchKernelGGL((fmha_d64<QS, NW, PART>), grid, dim3(64 * NW), 0, stream, p);
}

}  // namespace
}  // namespace h3v

using namespace h3v;

static int attention_common(const char* what, const uint16_t* q, int64_t q_token_stride, int64_t q_head_stride, const uint16_t* k,
                            int64_t k_token_stride, int64_t k_head_stride, const uint16_t* v, int64_t v_token_stride,
                            int64_t v_head_stride, uint16_t* o, int64_t o_token_stride, int64_t o_head_stride,
                            int64_t batch, int64_t tokens, int64_t heads, float scale, bool may_split,
                            float* workspace, int64_t workspace_floats, hipStream_t stream) {
    H3V_REQUIRE(q && k && v && o, "%s: null pointer argument", what);
    H3V_REQUIRE(batch > 0 && tokens > 0 && heads > 0, "%s: batch, tokens and heads must be positive", what);
    H3V_REQUIRE(batch <= 65535 && heads <= 65535 && tokens <= (1 << 24), "%s: shape out of range", what);
    H3V_REQUIRE(scale > 0.0f && scale < 1e30f, "%s: scale must be positive and finite", what);
    const int64_t strides[8] = {q_token_stride, q_head_stride, k_token_stride, k_head_stride,
                                v_token_stride, v_head_stride, o_token_stride, o_head_stride};
    for (int i = 0; i < 8; ++i)
        H3V_REQUIRE(strides[i] > 0 && strides[i] % 8 == 0, "%s: token/head strides must be positive multiples of 8 "
                    "elements (16-byte rows)", what);
    H3V_REQUIRE(aligned(q, 16) && aligned(k, 16) && aligned(v, 16) && aligned(o, 8),
                "%s: q, k, v must be 16-byte and o 8-byte aligned", what);
    AttnParams p;
    p.q = q; p.k = k; p.v = v; p.o = o;
    p.q_ts = q_token_stride; p.q_hs = q_head_stride;
    p.k_ts = k_token_stride; p.k_hs = k_head_stride;
    p.v_ts = v_token_stride; p.v_hs = v_head_stride;
    p.o_ts = o_token_stride; p.o_hs = o_head_stride;
    p.tokens = (int)tokens;
    p.c = scale * 1.4426950408889634f;
    const AttnPlan plan = plan_attention(batch, tokens, heads, may_split, alone(stream));
    const int64_t floats = attention_ws_floats(plan, batch, tokens, heads);
    H3V_REQUIRE(floats == 0 || (workspace && workspace_floats >= floats && aligned(workspace, 16)),
                "%s: needs a 16-byte aligned workspace of %lld floats", what, (long long)floats);
    p.q_first = 0;
    p.splits = 1;
    p.split_blocks = plan.split_blocks;
    p.part = p.ml = nullptr;
    const int64_t head = plan.head;
    if (plan.shape == AttnShape::Q128) launch_fmha<1, 4, false>(p, head, heads, batch, stream);
    else if (plan.shape == AttnShape::Q256) launch_fmha<1, 8, false>(p, head, heads, batch, stream);
    else if (plan.shape == AttnShape::Q256x4) launch_fmha<2, 4, false>(p, head, heads, batch, stream);
    else launch_fmha<2, 8, false>(p, head, heads, batch, stream);
    const int64_t rest = tokens - head;
    if (rest > 0) {
        p.q_first = (int)head;
        if (plan.splits == 1) {
            launch_fmha<1, 8, false>(p, rest, heads, batch, stream);
        } else {
            const int64_t rows = batch * heads * rest;
            p.splits = plan.splits;
            p.part = workspace;
            p.ml = workspace + plan.splits * rows * kD;
            launch_fmha<1, 8, true>(p, rest, heads, batch, stream);
            hipLaunchKernelGGL(fmha_merge, dim3((unsigned)((rows * 16 + 255) / 256)), dim3(256), 0, stream, p, (int)heads,
                               rows);
        }
    }
    return launch_status(what);
}

extern "C" int h3v_attention_d64(const uint16_t* q, int64_t q_token_stride, int64_t q_head_stride, const uint16_t* k,
                                 int64_t k_token_stride, int64_t k_head_stride, const uint16_t* v,
                                 int64_t v_token_stride, int64_t v_head_stride, uint16_t* o, int64_t o_token_stride,
                                 int64_t o_head_stride, int64_t batch, int64_t tokens, int64_t heads, float scale,
                                 hipStream_t stream) {
    return attention_common("h3v_attention_d64", q, q_token_stride, q_head_stride, k, k_token_stride, k_head_stride, v,
                            v_token_stride, v_head_stride, o, o_token_stride, o_head_stride, batch, tokens, heads,
                            scale, false, nullptr, 0, stream);
}

extern "C" int64_t h3v_attention_d64_workspace_floats(int64_t batch, int64_t tokens, int64_t heads) {
    if (batch <= 0 || tokens <= 0 || heads <= 0 || batch > 65535 || heads > 65535 || tokens > (1 << 24)) return 0;
    // a split does not depend on the stream
    return attention_ws_floats(plan_attention(batch, tokens, heads, true, true), batch, tokens, heads);
}

extern "C" int h3v_attention_d64_ws(const uint16_t* q, int64_t q_token_stride, int64_t q_head_stride, const uint16_t* k,
                                    int64_t k_token_stride, int64_t k_head_stride, const uint16_t* v,
                                    int64_t v_token_stride, int64_t v_head_stride, uint16_t* o,
                                    int64_t o_token_stride, int64_t o_head_stride, int64_t batch, int64_t tokens,
                                    int64_t heads, float scale, float* workspace, int64_t workspace_floats,
                                    hipStream_t stream) {
    return attention_common("h3v_attention_d64_ws", q, q_token_stride, q_head_stride, k, k_token_stride, k_head_stride,
                            v, v_token_stride, v_head_stride, o, o_token_stride, o_head_stride, batch, tokens, heads,
                            scale, true, workspace, workspace_floats, stream);
}
