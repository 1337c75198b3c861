// Split-KV (flash-decoding) GQA decode for gfx950.
//
// Replaces the reference's decode_flash_gqa_bf16_kernel
// (src/cplusplus/FlashGQA/decode_flash_gqa_kernel.cu:119-389), which walks the
// whole sequence serially per (kv head, batch) workgroup.  Here:
//   pass 1 (decode_split_kernel): 4 waves per (split of the KV sequence,
//     kv head, batch), two such items (adjacent kv heads) per 8-wave
//     workgroup when the kv heads pair up.  Each wave streams 32-token steps;
//     every K/V byte is read once from HBM and serves all G query heads of
//     the group.
//       K and V rows stream in with coalesced 16-byte non-temporal loads
//       (a quarter-wave reads one 256-byte row) and are staged in LDS
//       S^T[t][h] = K[t][:] . Q[h][:]        v_mfma_f32_16x16x32_bf16
//       online softmax in fp32 (exp2 with log2(e) folded into the scale), P
//       rounded to bf16 before P.V and the rowsum kept from the fp32 P, as the
//       reference does (decode_flash_gqa_kernel.cu:266-278)
//       O^T[d][h] += V^T[d][t] . P^T[t][h]   v_mfma_f32_16x16x32_bf16, V^T
//                                            read transposed from the staged
//                                            rows (ds_read_b64_tr_b16)
//     The 4 waves merge their (max, sum, O) in LDS; with one split the
//     workgroup writes the normalised bf16 output directly, otherwise it
//     writes an fp32 partial (O, max, sum) to the workspace.
//     Ragged batches share their tokens out evenly over the chip instead
//     (decode_list_kernel).
//   pass 2 (decode_combine_kernel): log-sum-exp merge of the partials.
//
// Paged KV cache (fgqa_decode_paged): the same kernels read K/V rows through a
// block table (token t of sequence b lives in page block_table[b][t / page],
// slot t % page), in bf16 or in OCP fp8 e4m3 with per-tensor scales.  fp8 rows
// are widened to bf16 exactly (v_cvt_scalef32_pk_bf16_fp8, scale 1) as they are
// staged in LDS; the K scale is folded into the softmax scale and the V scale
// into the output, so the arithmetic after staging is the bf16 path's.  Pages
// of at least one load instruction's rows (4 bf16 rows, 8 fp8 rows) are read
// by page segment (min(page, 32) rows of a step): one buffer resource per
// segment, the wave's pages taken from one vector load of the block table per
// 64 segments; smaller pages, and caches whose page bytes reach 2^31, look up
// each row's page and form its 64-bit address.
#include <math.h>

#include "fgqa_device.h"
#include "fgqa_internal.h"

namespace fgqa {

struct DecodeParams {
    const __bf16* q;
    const __bf16* k;
    const __bf16* v;
    __bf16* o;
    float* lse;
    const int32_t* seqlens;
    float* part_o;   // [B, Hkv, nsplit, G, 128]
    float* part_ml;  // [B, Hkv, nsplit, G, 2]  (max in log2 units, sum)
    int64_t q_sb, q_sh;
    int64_t k_sb, k_ss, k_sh;
    int64_t v_sb, v_ss, v_sh;
    int64_t o_sb, o_sh;
    const int32_t* work;   // ragged work list: [0] = entries, then (b << 16 | split) per entry; or null
    int64_t* prefix;       // teams: [B + 1] 128-token blocks before each sequence, then their total
    int teams;             // > 0: the ragged batch's blocks are shared out evenly over this many teams
    int batch, max_seqlen, hq, hkv, group;
    int nsplit, chunk;
    float scale_log2;
    // paged KV: k/v are the page caches, strides {page, slot, head} in elements
    // of the cache type; page of token t = block_table[b * bt_stride + (t >> page_shift)]
    const int32_t* block_table;
    int64_t bt_stride;
    int page_shift;
    int num_pages;      // page indices are clamped to [0, num_pages)
    float v_scale;      // multiplies O (the fp8 V scale; 1 otherwise)
};

// Cache layouts the decode items read.
enum DecKv { kKvContig = 0, kKvPagedBf16 = 1, kKvPagedFp8 = 2 };

// 16 OCP fp8 e4m3 values -> 16 bf16 (exact: every e4m3 value is a bf16 value).
__device__ __forceinline__ void fp8x16_to_bf16(u32x4_t in, u32x4_t* lo, u32x4_t* hi) {
    uint32_t w[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        w[2 * i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(in[i], 1.0f, false));
        w[2 * i + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(in[i], 1.0f, true));
    }
    *lo = u32x4_t{w[0], w[1], w[2], w[3]};
    *hi = u32x4_t{w[4], w[5], w[6], w[7]};
}

constexpr int kDecThreads = 256;
constexpr int kDecWaves = kDecThreads / kWave;
constexpr int kDecStep = 32;        // tokens per wave step (two 16-token MFMA blocks)
constexpr int kDecRowStride = 136;  // LDS row stride (elements) of a staged K or V row: 272 B
                                    // spreads 16 rows over all 64 banks for b128 reads
constexpr int kDecTileElems = kDecStep * kDecRowStride;
constexpr int kDecSmemBytes = kDecWaves * 2 * kDecTileElems * 2;  // per wave: K tile + V tile
static_assert(kDecWaves * 16 * kHeadDim * 4 + kDecWaves * 16 * 2 * 4 <= kDecSmemBytes,
              "wave merge buffers must fit in the staging area");

__device__ __forceinline__ int clamp_len(const DecodeParams& p, int b) {
    int len = p.seqlens ? p.seqlens[b] : p.max_seqlen;
    return min(max(len, 0), p.max_seqlen);
}

// One item of pass 1: tokens [t_begin, t_end) (not empty) of one sequence and
// kv head, run by 4 waves (tid: the thread's index among them, smem: their
// kDecSmemBytes of LDS).  whole: the item is the sequence's only one and
// writes O and the LSE; otherwise its fp32 partial goes to rows slot0 + head
// of the workspace.  kSeg (paged
// caches, 0 or a power of two from one load instruction's rows up to 32): the
// rows of a 32-token step fall into page segments of kSeg rows
// (kSeg = min(page, 32)), each read through one buffer resource; 0 is the
// general form, with a page lookup and a 64-bit address per row.
// The only workgroup barriers are the two of the wave merge, so two items of
// the same tokens can share a workgroup.
template <int kKv, int kSeg = 0>
__device__ __forceinline__ void dec_item(const DecodeParams& p, unsigned char* smem, int t_begin, int t_end, int kvh,
                                         int b, int tid, bool whole, int64_t slot0) {
    const int lane = tid & (kWave - 1);
    constexpr bool kUni = kSeg > 0;
    const int wave = kUni ? __builtin_amdgcn_readfirstlane(tid / kWave) : tid / kWave;
    const int l16 = lane & 15;
    const int g4 = lane >> 4;

    __bf16* kl = reinterpret_cast<__bf16*>(smem) + wave * 2 * kDecTileElems;
    __bf16* vl = kl + kDecTileElems;

    // Q^T as the B operand: lane holds Q[h = l16][32*kk + 8*g4 .. +7]; heads >= G are zero.
    bf16x8_t qop[4];
    {
        const bool hv = l16 < p.group;
        const __bf16* qrow = p.q + b * p.q_sb + (int64_t)(kvh * p.group + (hv ? l16 : 0)) * p.q_sh;
        const u32x4_t zero = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            u32x4_t t = *reinterpret_cast<const u32x4_t*>(qrow + kk * 32 + g4 * 8);
            qop[kk] = as_bf16x8(hv ? t : zero);
        }
    }

    float m_run = -INFINITY;
    float l_run = 0.f;  // this lane's share of the rowsum of head l16
    f32x4_t oacc[8];
#pragma unroll
    for (int db = 0; db < 8; ++db) oacc[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    const int n_steps = (t_end - t_begin + kDecStep - 1) / kDecStep;
    // One step = 32 token rows of K and of V.  bf16: load r (0..7) of a lane
    // covers row 4*r + g4, 16-byte chunk l16, so each quarter-wave reads one
    // whole 256-byte row (the coalesced pattern).  fp8: rows are 128 bytes;
    // load r (0..3) covers row 8*r + lane/8, chunk lane%8.
    constexpr int kRows = (kKv == kKvPagedFp8) ? 4 : 8;
    const int fp8_row = lane >> 3;
    const int fp8_chunk = lane & 7;
    auto row_of = [&](int r) { return (kKv == kKvPagedFp8) ? 8 * r + fp8_row : 4 * r + g4; };
    u32x4_t kreg[kRows];
    u32x4_t vreg[kRows];

    // Contiguous cache: buffer resources end at the split's last valid token,
    // so later tokens read as zero.
    const uint32_t kss = (uint32_t)(p.k_ss * 2);
    const uint32_t vss = (uint32_t)(p.v_ss * 2);
    __amdgpu_buffer_rsrc_t krs, vrs;
    if constexpr (kKv == kKvContig) {
        krs = make_rsrc(p.k + b * p.k_sb + kvh * p.k_sh, (uint32_t)(t_end - 1) * kss + kHeadDim * 2);
        vrs = make_rsrc(p.v + b * p.v_sb + kvh * p.v_sh, (uint32_t)(t_end - 1) * vss + kHeadDim * 2);
    }
    // Paged cache: each row's page comes from the block table one step ahead
    // of its load.  Tokens past the split's end reuse its last token (their
    // scores are masked; the row only has to be finite).
    constexpr int kElemBytes = (kKv == kKvPagedFp8) ? 1 : 2;
    const unsigned char* kbase = reinterpret_cast<const unsigned char*>(p.k) + kvh * p.k_sh * kElemBytes;
    const unsigned char* vbase = reinterpret_cast<const unsigned char*>(p.v) + kvh * p.v_sh * kElemBytes;
    const int32_t* bt = p.block_table + (int64_t)b * p.bt_stride;
    const int pmask = (1 << p.page_shift) - 1;
    int pg[kRows];
    // kSeg > 0: segment g of a step (rows kSeg*g .. +kSeg-1, one page) is
    // read through one buffer resource per cache, starting at the segment's
    // first row and ending at the split's last token (rows past it read as
    // zeros).  The wave's segment pages come 64 at a time from one vector
    // load of the block table (lane l: the wave's segment pt_first + l, its
    // segments numbered n * kSegs + g for its n-th step) and are taken out
    // with v_readlane (a scalar load would share its wait counter with the
    // LDS traffic).  Load instruction i
    // of a segment reads its rows kR*i .. kR*i + kR - 1 at a per-lane offset
    // that is the same in every segment and step.  The host picks kSeg only
    // when a page's bytes stay below 2^31.
    constexpr int kR = (kKv == kKvPagedFp8) ? 8 : 4;           // rows per load instruction
    constexpr int kSegs = kUni ? kDecStep / kSeg : 1;          // segments per step
    constexpr int kPerSeg = kRows / kSegs;                     // load instructions per segment
    static_assert(!kUni || (kSeg >= kR && kSeg <= kDecStep && kPerSeg * kSegs == kRows), "page segment");
    constexpr uint32_t kRowBytes = kHeadDim * kElemBytes;
    const uint32_t kss_e = (uint32_t)(p.k_ss * kElemBytes);
    const uint32_t vss_e = (uint32_t)(p.v_ss * kElemBytes);
    const int64_t ksb_e = p.k_sb * kElemBytes;
    const int64_t vsb_e = p.v_sb * kElemBytes;
    const int t_end_u = kUni ? __builtin_amdgcn_readfirstlane(t_end) : t_end;
    [[maybe_unused]] uint32_t kvoff[kPerSeg], vvoff[kPerSeg];
    if constexpr (kUni) {
        const int lr = (kKv == kKvPagedFp8) ? fp8_row : g4;             // the lane's row in an instruction
        const int cb = (kKv == kKvPagedFp8) ? fp8_chunk * 16 : l16 * 16;
#pragma unroll
        for (int i = 0; i < kPerSeg; ++i) {
            kvoff[i] = (uint32_t)(kR * i + lr) * kss_e + cb;
            vvoff[i] = (uint32_t)(kR * i + lr) * vss_e + cb;
        }
    }
    [[maybe_unused]] int pt_lane = 0;       // block table entry of segment pt_first + lane
    [[maybe_unused]] int pt_first = -kWave;
    [[maybe_unused]] auto pt_load = [&](int first) {
        const int n = first + lane;
        const int tok = min(t_begin + (wave + kDecWaves * (n / kSegs)) * kDecStep + kSeg * (n % kSegs), t_end_u - 1);
        pt_lane = bt[tok >> p.page_shift];
        pt_first = first;
    };
    if constexpr (kUni) pt_load(0);
    auto fetch_pages = [&](int s) {
        if constexpr (kUni) {
            (void)s;   // the pages are taken out in load_step
        } else if constexpr (kKv != kKvContig) {
            // Raw entries: they are clamped where load_step uses them.  A
            // clamp here would make the wave wait for the table loads at once,
            // and vector loads complete in order, so that wait would also take
            // the K/V loads issued just before, leaving none in flight while
            // the step computes.
#pragma unroll
            for (int r = 0; r < kRows; ++r) {
                const int tok = min(t_begin + s * kDecStep + row_of(r), t_end - 1);
                pg[r] = bt[tok >> p.page_shift];
            }
        }
    };
    auto load_step = [&](int s) {
        const int t0 = t_begin + s * kDecStep;
        if constexpr (kUni) {
            const int n0 = ((s - wave) / kDecWaves) * kSegs;   // the wave's first segment of step s
            if (n0 + kSegs > pt_first + kWave) pt_load(n0);
#pragma unroll
            for (int g = 0; g < kSegs; ++g) {
                pg[g] = min(max(__builtin_amdgcn_readlane(pt_lane, n0 - pt_first + g), 0), p.num_pages - 1);
            }
#pragma unroll
            for (int g = 0; g < kSegs; ++g) {
                const int tok = t0 + kSeg * g;
                const int nv = min(kSeg, t_end_u - tok);   // rows before the split's end
                const uint32_t slot = (uint32_t)(tok & pmask);
                const __amdgpu_buffer_rsrc_t kr = make_rsrc(kbase + pg[g] * ksb_e + slot * kss_e,
                                                            nv > 0 ? (uint32_t)(nv - 1) * kss_e + kRowBytes : 0u);
                const __amdgpu_buffer_rsrc_t vr = make_rsrc(vbase + pg[g] * vsb_e + slot * vss_e,
                                                            nv > 0 ? (uint32_t)(nv - 1) * vss_e + kRowBytes : 0u);
#pragma unroll
                for (int i = 0; i < kPerSeg; ++i) {
                    kreg[g * kPerSeg + i] = buf_load16_nt(kr, kvoff[i]);
                    vreg[g * kPerSeg + i] = buf_load16_nt(vr, vvoff[i]);
                }
            }
        } else if constexpr (kKv == kKvContig) {
#pragma unroll
            for (int r = 0; r < 8; ++r) kreg[r] = buf_load16_nt(krs, (uint32_t)(t0 + r * 4 + g4) * kss + l16 * 16);
#pragma unroll
            for (int r = 0; r < 8; ++r) vreg[r] = buf_load16_nt(vrs, (uint32_t)(t0 + r * 4 + g4) * vss + l16 * 16);
        } else {
            const int cb = (kKv == kKvPagedFp8) ? fp8_chunk * 16 : l16 * 16;
#pragma unroll
            for (int r = 0; r < kRows; ++r) {
                const int slot = min(t0 + row_of(r), t_end - 1) & pmask;
                const int page = min(max(pg[r], 0), p.num_pages - 1);
                const int64_t ko = ((int64_t)page * p.k_sb + (int64_t)slot * p.k_ss) * kElemBytes + cb;
                const int64_t vo = ((int64_t)page * p.v_sb + (int64_t)slot * p.v_ss) * kElemBytes + cb;
                kreg[r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(kbase + ko));
                vreg[r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(vbase + vo));
            }
        }
    };

    int st = wave;
    if (st < n_steps) {
        fetch_pages(st);
        load_step(st);
    }
    if (st + kDecWaves < n_steps) fetch_pages(st + kDecWaves);
    for (; st < n_steps; st += kDecWaves) {
        // Stage this step's rows (fp8 widened to bf16), then put the next
        // step's loads and the page lookups of the step after in flight.
        if constexpr (kKv == kKvPagedFp8) {
#pragma unroll
            for (int r = 0; r < kRows; ++r) {
                u32x4_t lo, hi;
                __bf16* kd = kl + row_of(r) * kDecRowStride + fp8_chunk * 16;
                __bf16* vd = vl + row_of(r) * kDecRowStride + fp8_chunk * 16;
                fp8x16_to_bf16(kreg[r], &lo, &hi);
                *reinterpret_cast<u32x4_t*>(kd) = lo;
                *reinterpret_cast<u32x4_t*>(kd + 8) = hi;
                fp8x16_to_bf16(vreg[r], &lo, &hi);
                *reinterpret_cast<u32x4_t*>(vd) = lo;
                *reinterpret_cast<u32x4_t*>(vd + 8) = hi;
            }
        } else {
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                *reinterpret_cast<u32x4_t*>(kl + (r * 4 + g4) * kDecRowStride + l16 * 8) = kreg[r];
                *reinterpret_cast<u32x4_t*>(vl + (r * 4 + g4) * kDecRowStride + l16 * 8) = vreg[r];
            }
        }
        if (st + kDecWaves < n_steps) load_step(st + kDecWaves);
        if (st + 2 * kDecWaves < n_steps) fetch_pages(st + 2 * kDecWaves);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

        // S^T = K Q^T; K as the A operand: lane holds K[16*tb + l16][32*kk + 8*g4 .. +7].
        const int t0 = t_begin + st * kDecStep;
        f32x4_t s[2];
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            s[tb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const bf16x8_t ka =
                    *reinterpret_cast<const bf16x8_t*>(kl + (tb * 16 + l16) * kDecRowStride + kk * 32 + g4 * 8);
                s[tb] = mfma16(ka, qop[kk], s[tb]);
            }
        }

        // Online softmax for head l16 over tokens t0 + 16*tb + 4*g4 + i.
        float x[8];
        float tmax = -INFINITY;
#pragma unroll
        for (int tb = 0; tb < 2; ++tb)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int tok = t0 + tb * 16 + g4 * 4 + i;
                const float val = (tok < t_end) ? s[tb][i] * p.scale_log2 : -INFINITY;
                x[tb * 4 + i] = val;
                tmax = fmaxf(tmax, val);
            }
        tmax = xor_max(xor_max(tmax, 16), 32);
        const float m_new = fmaxf(m_run, tmax);  // finite: every step holds a valid token
        const float alpha = fast_exp2(m_run - m_new);
        float psum = 0.f;
        bf16x8_t pop;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float pv = fast_exp2(x[j] - m_new);
            psum += pv;
            pop[j] = (__bf16)pv;
        }
        l_run = l_run * alpha + psum;
        m_run = m_new;
#pragma unroll
        for (int db = 0; db < 8; ++db) oacc[db] *= alpha;

        // V^T as the A operand: lane holds V[token(slot)][16*db + l16] for the
        // 8 slots of group g4: tokens 4*g4 + {0..3} and 16 + 4*g4 + {0..3},
        // the same tokens whose P this lane already holds.  Two transposed
        // reads (ds_read_b64_tr_b16) per column block: source lane l16 of the
        // group points at row 4*g4 + l16/4 (+16), columns 16*db + 4*(l16%4) .. +3.
        const __bf16* vsrc = vl + (4 * g4 + (l16 >> 2)) * kDecRowStride + 4 * (l16 & 3);
#pragma unroll
        for (int db = 0; db < 8; ++db) {
            const bf16x4_t lo = lds_read_tr16(vsrc + db * 16);
            const bf16x4_t hi = lds_read_tr16(vsrc + 16 * kDecRowStride + db * 16);
            oacc[db] = mfma16(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), pop, oacc[db]);
        }

        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

    l_run = xor_sum(xor_sum(l_run, 16), 32);

    // Merge the 4 waves in LDS (reusing the staging area).
    __syncthreads();
    float* ow = reinterpret_cast<float*>(smem);        // [wave][16][128]
    float* mlw = ow + kDecWaves * 16 * kHeadDim;       // [wave][16][2]
#pragma unroll
    for (int db = 0; db < 8; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i) ow[(wave * 16 + l16) * kHeadDim + db * 16 + g4 * 4 + i] = oacc[db][i];
    if (g4 == 0) {
        mlw[(wave * 16 + l16) * 2 + 0] = m_run;
        mlw[(wave * 16 + l16) * 2 + 1] = l_run;
    }
    __syncthreads();

    const int h = tid >> 4;
    const int d0 = (tid & 15) * 8;
    if (h >= p.group) return;
    float mw[kDecWaves];
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < kDecWaves; ++w) {
        mw[w] = mlw[(w * 16 + h) * 2];
        M = fmaxf(M, mw[w]);
    }
    float L = 0.f;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kDecWaves; ++w) {
        const float c = (mw[w] == -INFINITY) ? 0.f : fast_exp2(mw[w] - M);
        L += c * mlw[(w * 16 + h) * 2 + 1];
        const float* src = ow + (w * 16 + h) * kHeadDim + d0;
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] += c * src[j];
    }
    const int qh = kvh * p.group + h;
    if (whole) {
        const float inv = p.v_scale / L;
        bf16x8_t out;
#pragma unroll
        for (int j = 0; j < 8; ++j) out[j] = (__bf16)(acc[j] * inv);
        *reinterpret_cast<bf16x8_t*>(p.o + b * p.o_sb + qh * p.o_sh + d0) = out;
        if (p.lse != nullptr && (tid & 15) == 0) p.lse[(int64_t)b * p.hq + qh] = M * kLn2 + logf(L);
    } else {
        const int64_t slot = slot0 + h;
        float* po = p.part_o + slot * kHeadDim + d0;
        const float vs = p.v_scale;
        *reinterpret_cast<f32x4_t*>(po) = f32x4_t{acc[0] * vs, acc[1] * vs, acc[2] * vs, acc[3] * vs};
        *reinterpret_cast<f32x4_t*>(po + 4) = f32x4_t{acc[4] * vs, acc[5] * vs, acc[6] * vs, acc[7] * vs};
        if ((tid & 15) == 0) {
            p.part_ml[slot * 2 + 0] = M;
            p.part_ml[slot * 2 + 1] = L;
        }
    }
}

// Pass 1 over the full (split, kv head, batch) grid.  kPair (an even number
// of kv heads): 8-wave workgroups over (split, kv head pair, batch), waves 0-3
// on kv head 2j and waves 4-7 on kv head 2j + 1, so that the two 256-byte
// pieces of a token's cache row that lie side by side are read together (at
// 480 four-wave workgroups 159.5 us, 240 eight-wave ones
// 145.4 us, outputs bit-identical).
template <bool kPair>
__global__ __launch_bounds__(kPair ? 2 * kDecThreads : kDecThreads) void decode_split_kernel(DecodeParams p) {
    __shared__ __attribute__((aligned(16))) unsigned char smem[(kPair ? 2 : 1) * kDecSmemBytes];
    const int half = kPair ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kDecThreads)) : 0;
    const int tid = (int)threadIdx.x - half * kDecThreads;
    const int kvh = kPair ? 2 * (int)blockIdx.y + half : blockIdx.y;
    const int split = blockIdx.x, b = blockIdx.z;
    const int len = clamp_len(p, b);
    const int t_begin = split * p.chunk;
    if (t_begin >= len) {
        // Empty split: the combine never reads it.  Without a combine pass an
        // empty sequence still needs its O = 0, lse = -inf written here.
        if (p.nsplit == 1 && (tid >> 4) < p.group) {
            const int qh = kvh * p.group + (tid >> 4);
            bf16x8_t z;
#pragma unroll
            for (int j = 0; j < 8; ++j) z[j] = (__bf16)0.f;
            *reinterpret_cast<bf16x8_t*>(p.o + b * p.o_sb + qh * p.o_sh + (tid & 15) * 8) = z;
            if (p.lse != nullptr && (tid & 15) == 0) p.lse[(int64_t)b * p.hq + qh] = -INFINITY;
        }
        return;
    }
    dec_item<kKvContig>(p, smem + half * kDecSmemBytes, t_begin, min(t_begin + p.chunk, len), kvh, b, tid,
                        p.nsplit == 1, (((int64_t)b * p.hkv + kvh) * p.nsplit + split) * p.group);
}

// Ragged batches with a split length given by the caller: build the work list
// of non-empty splits, full-length splits first and the partial last split of
// each sequence after them, longest first (batch order beyond kPlanSortMax
// sequences), so that equal work fills the GPU and the short items form the
// tail.  One workgroup; entry = (b << 16) | split, so batch < 2^15 and splits
// < 2^16 (checked on the host).
constexpr int kPlanThreads = 256;
constexpr int kPlanSortMax = 1024;   // remainders kept in LDS and length-sorted up to this batch size

// The value of the lane that DPP control kCtrl names, 0 where there is none or
// the row is not in kRows.
template <int kCtrl, int kRows, typename T>
__device__ __forceinline__ T dpp_or_0(T v) {
    if constexpr (sizeof(T) == 8) {
        const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)v, kCtrl, kRows, 0xF, true);
        const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), kCtrl, kRows, 0xF, true);
        return (T)(((uint64_t)hi << 32) | lo);
    } else {
        return __builtin_amdgcn_update_dpp(0, v, kCtrl, kRows, 0xF, true);
    }
}

// Folds each lane's value with those of all lanes before it (0: neutral): row
// shifts by 1, 2, 4 and 8, then the rows' last lanes broadcast to the rows
// after them.  (With LDS shuffles instead, two per step for a 64-bit sum, a
// ragged decode of 13 us took 0.3 us longer.)
template <typename T, typename F>
__device__ __forceinline__ T wave_fold(T v, F&& f) {
    v = f(v, dpp_or_0<0x111, 0xF>(v));
    v = f(v, dpp_or_0<0x112, 0xF>(v));
    v = f(v, dpp_or_0<0x114, 0xF>(v));
    v = f(v, dpp_or_0<0x118, 0xF>(v));
    v = f(v, dpp_or_0<0x142, 0xA>(v));
    return f(v, dpp_or_0<0x143, 0xC>(v));
}

// Exclusive prefix sum of one value per thread over a workgroup of kThreads.
// kAgain: another scan in s_wave follows (else a barrier does before s_wave's
// memory is written again).
template <int kThreads, bool kAgain, typename T>
__device__ __forceinline__ T block_exclusive_scan(T v, T* s_wave, T* total) {
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const T incl = wave_fold(v, [](T a, T b) { return a + b; });
    if (lane == kWave - 1) s_wave[wave] = incl;
    __syncthreads();
    T base = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kThreads / kWave; ++w) {
        base += (w < wave) ? s_wave[w] : 0;
        all += s_wave[w];
    }
    if constexpr (kAgain) __syncthreads();
    *total = all;
    return base + incl - v;
}

__global__ __launch_bounds__(kPlanThreads) void decode_plan_kernel(DecodeParams p, int32_t* work) {
    __shared__ int s_wave[kPlanThreads / kWave];
    __shared__ int s_rem[kPlanSortMax];   // len % chunk per sequence (batch <= kPlanSortMax)
    const int tid = threadIdx.x;
    const bool sort = p.batch <= kPlanSortMax;
    // sequences b = tid, tid + 256, ... belong to this thread
    int nf = 0, np = 0;
    for (int b = tid; b < p.batch; b += kPlanThreads) {
        const int len = clamp_len(p, b);
        nf += len / p.chunk;
        np += (len % p.chunk) != 0;
        if (sort) s_rem[b] = len % p.chunk;
    }
    int n_full, n_part;
    int pos_f = block_exclusive_scan<kPlanThreads, true>(nf, s_wave, &n_full);
    int pos_p = block_exclusive_scan<kPlanThreads, true>(np, s_wave, &n_part);   // also publishes s_rem (barriers inside)
    if (tid == 0) work[0] = n_full + n_part;
    for (int b = tid; b < p.batch; b += kPlanThreads) {
        const int len = clamp_len(p, b);
        const int full = len / p.chunk;
        for (int sp = 0; sp < full; ++sp) work[1 + pos_f + sp] = (b << 16) | sp;
        pos_f += full;
        const int rem = len % p.chunk;
        if (rem == 0) continue;
        int rank = pos_p;   // batch order
        if (sort) {
            rank = 0;       // longest remainder first, ties by batch
            for (int o = 0; o < p.batch; ++o) {
                const int ro = s_rem[o];
                rank += (ro > rem) || (ro == rem && o < b);
            }
        }
        work[1 + n_full + rank] = (b << 16) | full;
        ++pos_p;
    }
    // Without a combine pass, empty sequences (no list entry) still need
    // O = 0 and lse = -inf.
    if (p.nsplit == 1) {
        for (int b = 0; b < p.batch; ++b) {
            if (clamp_len(p, b) != 0) continue;
            for (int i = tid; i < p.hq * 16; i += kPlanThreads) {
                const int qh = i >> 4;
                bf16x8_t z;
#pragma unroll
                for (int j = 0; j < 8; ++j) z[j] = (__bf16)0.f;
                *reinterpret_cast<bf16x8_t*>(p.o + b * p.o_sb + qh * p.o_sh + (i & 15) * 8) = z;
                if (p.lse != nullptr && (i & 15) == 0) p.lse[(int64_t)b * p.hq + qh] = -INFINITY;
            }
        }
    }
}

// Pass 1 over a ragged batch.  A sequence is a run of 128-token blocks (one
// pass of 4 waves); team t of n takes blocks [total * t / n, total * (t + 1) /
// n) of the concatenated sequences, one workgroup per kv head or head pair, so
// every CU streams the same number of tokens whatever the lengths, and the
// workgroups of a team read the same rows side by side.  A team's range is cut
// at the sequences' ends into items; a sequence inside one range is written
// directly, and only the (at most two per team) items of a sequence that
// crosses a range's end leave partials: slot 2t for one that starts inside the
// sequence, 2t + 1 for the sequence's first.  Each workgroup finds its range
// by itself from the lengths (a scan of one value per thread), which needs no
// planning launch before it.  Against 4096-token splits handed out by a
// planning kernel's work list: 8 sequences of up to 6000 tokens, Hq = 32,
// Hkv = 8, bf16 pages: 88.5 -> 30.3 us; 64 of up to 32768, Hq = 64, fp8 pages:
// 395.8 -> 360.9 us.
//
// Cutting sequences costs a second item per team and the combine.  Where whole
// sequences are nearly as even (kWholeSlack), a team takes `per` of them in a
// row, and nothing is left to combine.
//
// A split length given by the caller keeps the work list (p.work): a fixed
// grid walks its entries, each once per kv head or pair (the head fastest, so
// heads of one split run together).
//
// kPair (an even number of kv heads): 8-wave workgroups, waves 0-3 on kv head
// 2j and waves 4-7 on kv head 2j + 1 of the same tokens.  Each half reads its
// own head's rows, but the two halves' loads of one token arrive together, so
// the 2 x 128-byte (fp8) or 2 x 256-byte (bf16) pieces of a cache row that lie
// side by side in memory are read at the same time: a streaming read of
// config 3's fp8 page pattern ran at 5.84 TB/s with one head per workgroup and
// 6.45 TB/s with head pairs.  Both halves of a workgroup hold the same tokens
// of the same sequence, so they pass the same workgroup barriers.
__device__ __forceinline__ int64_t team_start(int64_t total, int teams, int t) { return total * t / teams; }

// Teams that get blocks: every one of them at least one.
__device__ __forceinline__ int team_count(const DecodeParams& p, int64_t total) {
    return total < p.teams ? (int)total : p.teams;
}

// Blocks per team that the cuts cost: a team runs per = ceil(batch / teams)
// whole sequences if per times the longest one is at most this much above an
// even share, unless the batch has a block per team or less.  Equal lengths,
// us cut / whole: 60 of 4096 (Hq = 128, Hkv = 8) 170.6 / 155.7; Hq = 32,
// Hkv = 8, 16-token pages: 60 of 1024 48.9 / 43.0, 20 of 512 (2.75 above)
// 21.6 / 17.8, but 20 of 1024 (5.5 above) 26.7 / 30.0; 2 of 512 with Hq = 16,
// Hkv = 2 (8 blocks, 256 teams) 13.9 / 15.5.
constexpr int kWholeSlack = 4;
// The prefix's total then.
constexpr int64_t kWholeTeams = -1;

__device__ __forceinline__ int seq_blocks(int len) {
    return (len + plan::kDecodeStepRound - 1) / plan::kDecodeStepRound;
}

template <int kKv, int kSeg = 0, bool kPair = false>
__global__ __launch_bounds__(kPair ? 2 * kDecThreads : kDecThreads) void decode_list_kernel(DecodeParams p) {
    constexpr int kThreads = kPair ? 2 * kDecThreads : kDecThreads;
    __shared__ __attribute__((aligned(16))) unsigned char smem[(kPair ? 2 : 1) * kDecSmemBytes];
    // wave-uniform (readfirstlane), so the buffer resources built from the
    // head stay scalar
    const int half = kPair ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kDecThreads)) : 0;
    const int per_entry = kPair ? p.hkv / 2 : p.hkv;
    const int tid = (int)threadIdx.x - half * kDecThreads;
    // work list: items blockIdx.x, + gridDim.x, ...
    int item = blockIdx.x;
    const int n_items = p.work != nullptr ? p.work[0] * per_entry : 0;
    // teams: blocks [g0, g1) of the batch, the first of them block `blk` of
    // sequence b, and none of sequence b_end
    const int team = blockIdx.x / per_entry;
    int64_t g0 = 0, g1 = 0;
    int b = 0, b_end = p.batch, blk = 0;
    if (p.work == nullptr) {
        int64_t* s_wave = reinterpret_cast<int64_t*>(smem);
        int* s_pos = reinterpret_cast<int*>(s_wave + kThreads / kWave);
        int* s_max = s_pos + 2;   // per wave
        const int per = (p.batch + kThreads - 1) / kThreads;
        const int b_lo = min((int)threadIdx.x * per, p.batch), b_hi = min(b_lo + per, p.batch);
        int64_t sum = 0, total;
        int longest = 0;
        for (int i = b_lo; i < b_hi; ++i) {
            const int n = seq_blocks(clamp_len(p, i));
            sum += n;
            longest = max(longest, n);
        }
        longest = wave_fold(longest, [](int x, int y) { return max(x, y); });   // (all of it in the last lane)
        if ((threadIdx.x & (kWave - 1)) == kWave - 1) s_max[threadIdx.x / kWave] = longest;   // published by the scan's barrier
        int64_t at = block_exclusive_scan<kThreads, false>(sum, s_wave, &total);
        // (uniform: the compiler does not see it through the LDS sum)
        total = (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(total >> 32)) << 32) |
                          (uint32_t)__builtin_amdgcn_readfirstlane((int)total));
        longest = 0;
#pragma unroll
        for (int w = 0; w < kThreads / kWave; ++w) longest = max(longest, s_max[w]);
        longest = __builtin_amdgcn_readfirstlane(longest);
        const int whole_per = (p.batch + p.teams - 1) / p.teams;
        const bool whole_seqs = total > p.teams && (int64_t)whole_per * longest * p.teams <=
                                                        total + (int64_t)kWholeSlack * p.teams;
        if (blockIdx.x == 0 && threadIdx.x == 0) p.prefix[p.batch] = whole_seqs ? kWholeTeams : total;
        const int teams = team_count(p, total);
        if (whole_seqs) {
            b = min(team * whole_per, p.batch);
            b_end = min(b + whole_per, p.batch);
            g1 = total;   // (b_end ends the range)
        } else if (team < teams) {
            g0 = team_start(total, teams, team);
            g1 = team_start(total, teams, team + 1);
        }
        if (!whole_seqs) {
            const bool here = g0 >= at && g0 < at + sum;   // exactly one thread's, unless g0 is the end
            if (here || blockIdx.x == 0) {
                for (int i = b_lo; i < b_hi; ++i) {
                    const int n = seq_blocks(clamp_len(p, i));
                    if (blockIdx.x == 0) p.prefix[i] = at;
                    if (g0 >= at && g0 < at + n) {
                        s_pos[0] = i;
                        s_pos[1] = (int)(g0 - at);
                    }
                    at += n;
                }
            }
            if (g0 >= g1) return;
            __syncthreads();
            b = __builtin_amdgcn_readfirstlane(s_pos[0]);
            blk = __builtin_amdgcn_readfirstlane(s_pos[1]);
        }
    }
    while (true) {
        int kvh, t_begin, t_end;
        bool whole;
        int64_t slot;
        if (p.work != nullptr) {
            if (item >= n_items) break;
            const int e = p.work[1 + item / per_entry];
            kvh = item % per_entry;
            const int split = e & 0xffff;
            b = e >> 16;
            t_begin = split * p.chunk;
            t_end = min(t_begin + p.chunk, clamp_len(p, b));
            whole = p.nsplit == 1;
            kvh = kPair ? 2 * kvh + half : kvh;
            slot = ((int64_t)b * p.hkv + kvh) * p.nsplit + split;
            item += gridDim.x;
        } else {
            if (g0 >= g1 || b >= b_end) break;
            const int len = clamp_len(p, b);
            const int nb = seq_blocks(len);
            if (nb == 0) {   // empty sequences: the combine writes their O
                ++b;
                continue;
            }
            const int n = (int)min((int64_t)(nb - blk), g1 - g0);
            t_begin = blk * plan::kDecodeStepRound;
            t_end = min((blk + n) * plan::kDecodeStepRound, len);
            whole = n == nb;
            kvh = blockIdx.x % per_entry;
            kvh = kPair ? 2 * kvh + half : kvh;
            slot = (int64_t)(2 * team + (blk == 0 ? 1 : 0)) * p.hkv + kvh;
        }
        __syncthreads();   // the previous item's merge buffers alias the staging area
        dec_item<kKv, kSeg>(p, smem + half * kDecSmemBytes, t_begin, t_end, kvh, b, tid, whole, slot * p.group);
        if (p.work == nullptr) {
            g0 += (t_end - t_begin + plan::kDecodeStepRound - 1) / plan::kDecodeStepRound;
            ++b;
            blk = 0;
        }
    }
}

// Launches pass 1 over a ragged batch: the head-pair form (one 8-wave
// workgroup per CU) when the kv heads pair up, else two 4-wave workgroups per
// CU.  A work list's grid never exceeds what the CUs hold at once; the teams fill
// 256 CUs (kDecodeItemSlots), and on fewer they run in more than one round.
template <int kKv, int kSeg>
static void launch_list(const DecodeParams& p, int nsplit, int cus, hipStream_t s) {
    const bool pair = (p.hkv % 2) == 0;
    const int per_entry = pair ? p.hkv / 2 : p.hkv;
    const int64_t items = (int64_t)p.batch * nsplit * per_entry;   // most the list can hold
    const int64_t slots = (int64_t)(pair ? 1 : 2) * cus;
    const int grid = p.teams > 0 ? p.teams * per_entry : (int)(items < slots ? items : slots);
    if (pair)
        hipLaunchKernelGGL((decode_list_kernel<kKv, kSeg, true>), dim3(grid), dim3(2 * kDecThreads), 0, s, p);
    else
        hipLaunchKernelGGL((decode_list_kernel<kKv, kSeg, false>), dim3(grid), dim3(kDecThreads), 0, s, p);
}

// Log-sum-exp merge of the partials of each (sequence, query head): 16 lanes
// of 8 dims each x kWays ways, way w taking partials w, w + kWays, ... (in
// batches of kCombineBatch whose loads are all issued before any is used:
// slots past the last re-read it and are masked), then one merge of the ways
// through LDS.  A workgroup holds 16 / kWays heads.  The launch is bound by
// memory round trips, one per batch, so the host picks as many ways as one
// batch each needs (launch_combine).  With one way per head at 128 partials (one
// 32768-token sequence, Hq = 64, Hkv = 8): 27.4 us; 16 ways: 4.3 us.
template <bool kTeam, int kWays>
__global__ __launch_bounds__(kDecThreads) void decode_combine_kernel(DecodeParams p) {
    constexpr int kHeads = 16 / kWays;
    __shared__ float s_part[kWays > 1 ? kWays * kHeads * 16 * 10 : 1];   // acc[8], max, sum per lane
    const int b = blockIdx.y;
    const int d16 = threadIdx.x & 15;
    const int d0 = d16 * 8;
    const int way = (threadIdx.x >> 4) / kHeads;
    const int hl = (threadIdx.x >> 4) % kHeads;
    const int qh_raw = blockIdx.x * kHeads + hl;
    const int qh = min(qh_raw, p.hq - 1);   // lanes past the last head repeat it and store nothing
    const int kvh = qh / p.group;
    const int h = qh - kvh * p.group;
    const int len = clamp_len(p, b);
    // partial i: row base + i * step of the workspace (teams: the first one apart)
    int n;
    int64_t first, base, step;
    if constexpr (kTeam) {
        n = 0;
        first = base = step = 0;
        if (len > 0) {
            // (both loads before the test: one memory round trip)
            const int64_t total = p.prefix[p.batch], g0 = p.prefix[b], g1 = g0 + seq_blocks(len);
            asm volatile("" :: "s"(g0));
            if (total == kWholeTeams) return;   // the whole workgroup: pass 1 wrote every output
            const int teams = team_count(p, total);
            auto team_of = [&](int64_t g) {   // the last team whose start is at most g
                int t = (int)(g * teams / total);
                while (t + 1 < teams && team_start(total, teams, t + 1) <= g) ++t;
                return t;
            };
            const int t0 = team_of(g0), t1 = team_of(g1 - 1);
            if (t0 == t1) return;   // the whole workgroup: pass 1 wrote the sequence's output
            n = t1 - t0 + 1;
            first = ((int64_t)(2 * t0 + 1) * p.hkv + kvh) * p.group + h;
            step = (int64_t)2 * p.hkv * p.group;
            base = (int64_t)t0 * step + kvh * p.group + h;
        }
    } else {
        n = (len + p.chunk - 1) / p.chunk;
        step = p.group;
        first = base = ((int64_t)b * p.hkv + kvh) * p.nsplit * p.group + h;
    }
    __bf16* orow = p.o + b * p.o_sb + qh * p.o_sh + d0;
    const bool store = way == 0 && qh_raw < p.hq;
    if (n == 0) {   // (the whole workgroup)
        bf16x8_t z;
#pragma unroll
        for (int j = 0; j < 8; ++j) z[j] = (__bf16)0.f;
        if (store) *reinterpret_cast<bf16x8_t*>(orow) = z;
        if (store && p.lse != nullptr && d16 == 0) p.lse[(int64_t)b * p.hq + qh] = -INFINITY;
        return;
    }
    auto row_of = [&](int i) {
        const int c = min(i, n - 1);
        return c == 0 ? first : base + c * step;
    };
    constexpr int kCombineBatch = 8;
    float M = -INFINITY, L = 0.f;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int s0 = way; s0 < n; s0 += kCombineBatch * kWays) {
        float ms[kCombineBatch], ls[kCombineBatch];
        f32x4_t a[kCombineBatch], bb[kCombineBatch];
#pragma unroll
        for (int i = 0; i < kCombineBatch; ++i) {
            const int64_t slot = row_of(s0 + i * kWays);
            ms[i] = p.part_ml[slot * 2];
            ls[i] = p.part_ml[slot * 2 + 1];
            a[i] = *reinterpret_cast<const f32x4_t*>(p.part_o + slot * kHeadDim + d0);
            bb[i] = *reinterpret_cast<const f32x4_t*>(p.part_o + slot * kHeadDim + d0 + 4);
        }
        float m_new = M;
#pragma unroll
        for (int i = 0; i < kCombineBatch; ++i) m_new = fmaxf(m_new, ms[i]);
        const float c0 = (M == -INFINITY) ? 0.f : fast_exp2(M - m_new);
        L *= c0;
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] *= c0;
        M = m_new;
        // selects, not a branch, so the loads above stay ahead of every use
#pragma unroll
        for (int i = 0; i < kCombineBatch; ++i) {
            const bool valid = s0 + i * kWays < n;
            const float c = (ms[i] == -INFINITY) ? 0.f : fast_exp2(ms[i] - M);
            L = valid ? L + c * ls[i] : L;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc[j] = valid ? acc[j] + c * a[i][j] : acc[j];
                acc[4 + j] = valid ? acc[4 + j] + c * bb[i][j] : acc[4 + j];
            }
        }
    }
    if constexpr (kWays > 1) {
        // [way][head][value][lane]
        float* mine = s_part + (way * kHeads + hl) * 160 + d16;
#pragma unroll
        for (int j = 0; j < 8; ++j) mine[j * 16] = acc[j];
        mine[128] = M;
        mine[144] = L;
        __syncthreads();
        if (way != 0) return;
        const int nw = min(kWays, n);   // ways that held a partial
        const float m0 = M;
        for (int w = 1; w < nw; ++w) M = fmaxf(M, s_part[(w * kHeads + hl) * 160 + 128 + d16]);
        const float c0 = (m0 == -INFINITY) ? 0.f : fast_exp2(m0 - M);
        L *= c0;
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] *= c0;
        for (int w = 1; w < nw; ++w) {
            const float* o = s_part + (w * kHeads + hl) * 160 + d16;
            const float c = (o[128] == -INFINITY) ? 0.f : fast_exp2(o[128] - M);
            L += c * o[144];
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[j] += c * o[j * 16];
        }
    }
    if (!store) return;
    const float inv = 1.f / L;
    bf16x8_t out;
#pragma unroll
    for (int j = 0; j < 8; ++j) out[j] = (__bf16)(acc[j] * inv);
    *reinterpret_cast<bf16x8_t*>(orow) = out;
    if (p.lse != nullptr && d16 == 0) p.lse[(int64_t)b * p.hq + qh] = M * kLn2 + logf(L);
}

// Ways of the combine for `n` partials per (sequence, head): one batch of 8
// each, as far as 16 ways go (a ragged batch's n is the average sequence's,
// and a long one among short ones has more: 4 ways at least).
template <bool kTeam>
static void launch_combine(const DecodeParams& p, int64_t n, hipStream_t s) {
    if (n > 32)
        hipLaunchKernelGGL((decode_combine_kernel<kTeam, 16>), dim3(p.hq, p.batch), dim3(kDecThreads), 0, s, p);
    else if (kTeam || n > 8)
        hipLaunchKernelGGL((decode_combine_kernel<kTeam, 4>), dim3((p.hq + 3) / 4, p.batch), dim3(kDecThreads), 0, s,
                           p);
    else if constexpr (!kTeam)
        hipLaunchKernelGGL((decode_combine_kernel<false, 1>), dim3((p.hq + 15) / 16, p.batch), dim3(kDecThreads), 0, s,
                           p);
}

// The passes over a ragged batch (teams, or the work list of a given split length).
template <typename Launch>
static void run_ragged(const DecodeParams& p, int32_t* work, Launch&& pass1, hipStream_t s) {
    if (p.teams > 0) {
        pass1();
        // a sequence's share of the teams if it were the batch's average
        const int64_t blocks = ceil_div(p.max_seqlen, plan::kDecodeStepRound);
        const int64_t share = ceil_div(p.teams, p.batch) + 1;
        launch_combine<true>(p, share < blocks ? share : blocks, s);
        return;
    }
    hipLaunchKernelGGL(decode_plan_kernel, dim3(1), dim3(kPlanThreads), 0, s, p, work);
    pass1();
    if (p.nsplit > 1) launch_combine<false>(p, p.nsplit, s);
}

// One pass of the 4 decode waves covers the planner's split rounding.
static_assert(kDecWaves * kDecStep == plan::kDecodeStepRound, "decode split rounding");

namespace {
using plan::DecodePlan;
using plan::DecodeShape;

// Points p's partials, and the teams' prefix or the work list (returned, also
// in p.work), into the workspace.
int32_t* carve_workspace(const DecodePlan& plan, void* ws, DecodeParams* p) {
    char* w = static_cast<char*>(ws);
    if (plan.teams > 0) {
        p->teams = plan.teams;
        p->prefix = reinterpret_cast<int64_t*>(w + plan.team_prefix_off);
        p->part_o = reinterpret_cast<float*>(w);
        p->part_ml = reinterpret_cast<float*>(w + plan.team_ml_off);
        return nullptr;
    }
    if (plan.nsplit > 1) {
        p->part_o = reinterpret_cast<float*>(w);
        p->part_ml = reinterpret_cast<float*>(w + plan.part_o_bytes);
    }
    int32_t* work = plan.list ? reinterpret_cast<int32_t*>(w + plan.part_o_bytes + plan.part_ml_bytes) : nullptr;
    p->work = work;
    return work;
}

// The workspace of a call that needs one: the caller's (*ws, bytes), or for
// null and 0 the library's buffer, whose lock is then held.  Sets *ws, and the
// plan's form to what it holds.  A capture cannot grow the library's buffer: it
// takes the list's form where the buffer is large enough for that alone.
int take_workspace(DecodePlan* plan, size_t bytes, hipStream_t s, std::unique_lock<std::mutex>* lock, void** ws) {
    if (*ws == nullptr && bytes == 0) {
        *lock = workspace_lock();
        size_t want = plan->ws_bytes;
        const size_t have = internal_workspace_size();
        if (have < want && have >= plan->least_bytes) {
            hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
            if (hipStreamIsCapturing(s, &capture) != hipSuccess) (void)hipGetLastError();
            if (capture != hipStreamCaptureStatusNone) want = plan->least_bytes;
        }
        plan::fit_workspace(plan, want);
        int st = FGQA_OK;
        *ws = internal_workspace(want, &st);
        return st;
    }
    if (*ws == nullptr || bytes < plan->least_bytes) return FGQA_ERR_WORKSPACE;
    if (!aligned16(*ws)) return FGQA_ERR_UNSUPPORTED;
    plan::fit_workspace(plan, bytes);
    return FGQA_OK;
}

// The split plan of a validated call on the current device.
int plan_on_device(const DecodeShape& shape, DecodePlan* pl) {
    const int cus = plan::decode_needs_cus(shape) ? device_cu_count() : 0;
    return plan::plan_decode(shape, cus, pl);
}
}  // namespace
}  // namespace fgqa

using namespace fgqa;

extern "C" int fgqa_decode_workspace_bytes(const fgqa_decode_args* a, size_t* bytes) {
    if (bytes == nullptr) return FGQA_ERR_INVALID_ARGUMENT;
    int st = plan::validate_decode(a);
    if (st != FGQA_OK) return st;
    DecodePlan plan;
    st = plan_on_device(plan::decode_shape(a), &plan);
    if (st != FGQA_OK) return st;
    *bytes = plan.ws_bytes;
    return FGQA_OK;
}

// Device scratch of fgqa_decode_bf16_noalloc: the split partials and the
// ragged work list of one call (FGQA_DECODE_NOALLOC_SCRATCH_BYTES, held by
// every device the library runs on until the process ends).  In host code the
// name `scratch` is a host-side stand-in, not a device address: the address is
// looked up once per device (hipGetSymbolAddress, with that device current)
// and only that pointer is passed to kernels.
namespace fgqa {
namespace {
constexpr size_t kNoAllocScratchBytes = FGQA_DECODE_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];
constexpr int kScratchDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kScratchDevices] = {nullptr};

// The current device's copy of `scratch` (its address is looked up on the
// first call on that device).  Returns nullptr and sets *status on failure.
void* noalloc_scratch(int* status) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kScratchDevices) {
        *status = FGQA_ERR_HIP;
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void* ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || ptr == nullptr) {
            *status = FGQA_ERR_HIP;
            return nullptr;
        }
        g_scratch_ptr[dev] = ptr;
    }
    *status = FGQA_OK;
    return g_scratch_ptr[dev];
}

// The decode call; `noalloc`: the workspace is the device scratch above
// (the caller passes none), never the caller's or the library's buffer.
int decode_run(const fgqa_decode_args* a, void* stream, bool noalloc) {
    int st = plan::validate_decode(a);
    if (st != FGQA_OK) return st;
    st = plan::validate_decode_pointers(a);
    if (st != FGQA_OK) return st;
    if (a->batch == 0) return FGQA_OK;
    DecodePlan plan;
    st = plan_on_device(plan::decode_shape(a), &plan);
    if (st != FGQA_OK) return st;

    DecodeParams p;
    p.block_table = nullptr;
    p.bt_stride = 0;
    p.page_shift = 0;
    p.num_pages = 0;
    p.v_scale = 1.f;
    p.q = static_cast<const __bf16*>(a->q);
    p.k = static_cast<const __bf16*>(a->k);
    p.v = static_cast<const __bf16*>(a->v);
    p.o = static_cast<__bf16*>(a->o);
    p.lse = a->lse;
    p.seqlens = a->seqlens;
    p.part_o = nullptr;
    p.part_ml = nullptr;
    p.work = nullptr;
    p.prefix = nullptr;
    p.teams = 0;
    p.q_sb = a->q_stride[0];
    p.q_sh = a->q_stride[1];
    p.k_sb = a->k_stride[0];
    p.k_ss = a->k_stride[1];
    p.k_sh = a->k_stride[2];
    p.v_sb = a->v_stride[0];
    p.v_ss = a->v_stride[1];
    p.v_sh = a->v_stride[2];
    p.o_sb = a->o_stride[0];
    p.o_sh = a->o_stride[1];
    p.batch = a->batch;
    p.max_seqlen = a->max_seqlen;
    p.hq = a->num_q_heads;
    p.hkv = a->num_kv_heads;
    p.group = a->num_q_heads / a->num_kv_heads;
    p.nsplit = plan.nsplit;
    p.chunk = plan.chunk;
    p.scale_log2 = a->scale * kLog2e;

    const hipStream_t s = static_cast<hipStream_t>(stream);
    int32_t* work = nullptr;
    std::unique_lock<std::mutex> ws_lock;   // held through the launches when the library's buffer is used
    if (plan.ws_bytes > 0) {
        void* ws = a->workspace;
        if (noalloc) {
            // the partials and the list are written before they are read, so
            // the previous call's contents need no clearing
            if (plan.ws_bytes > kNoAllocScratchBytes) return FGQA_ERR_WORKSPACE;
            ws = noalloc_scratch(&st);
            if (ws == nullptr) return st;
        } else if (st = take_workspace(&plan, a->workspace_bytes, s, &ws_lock, &ws); st != FGQA_OK) {
            return st;
        }
        work = carve_workspace(plan, ws, &p);
    }

    if (a->max_seqlen == 0) {
        // Every sequence is empty: the combine writes O = 0, lse = -inf.
        launch_combine<false>(p, 1, s);
    } else if (plan.list) {
        const int cus = device_cu_count();
        if (cus <= 0) return FGQA_ERR_HIP;
        run_ragged(p, work, [&] { launch_list<kKvContig, 0>(p, plan.nsplit, cus, s); }, s);
    } else {
        // Head pairs once the grid holds at least one item per CU; smaller
        // grids are latency-bound and keep one item per workgroup (BASELINE
        // config 1's 16 items: 9.9 us paired, 9.4 us not).
        const int cus = device_cu_count();
        if (cus <= 0) return FGQA_ERR_HIP;
        const bool pair = p.hkv % 2 == 0 && (int64_t)p.nsplit * p.hkv * p.batch >= cus;
        if (pair)
            hipLaunchKernelGGL(decode_split_kernel<true>, dim3(p.nsplit, p.hkv / 2, p.batch), dim3(2 * kDecThreads), 0,
                               s, p);
        else
            hipLaunchKernelGGL(decode_split_kernel<false>, dim3(p.nsplit, p.hkv, p.batch), dim3(kDecThreads), 0, s, p);
        if (plan.nsplit > 1) launch_combine<false>(p, plan.nsplit, s);
    }
    if (hipGetLastError() != hipSuccess) return FGQA_ERR_HIP;
    return FGQA_OK;
}

}  // namespace
}  // namespace fgqa

extern "C" int fgqa_decode_bf16(const fgqa_decode_args* a, void* stream) { return decode_run(a, stream, false); }

extern "C" int fgqa_decode_bf16_noalloc(const fgqa_decode_args* a, void* stream) {
    if (a != nullptr && (a->workspace != nullptr || a->workspace_bytes != 0)) return FGQA_ERR_INVALID_ARGUMENT;
    return decode_run(a, stream, true);
}

// ---------------------------------------------------------------- paged KV cache
extern "C" int fgqa_decode_paged_workspace_bytes(const fgqa_decode_paged_args* a, size_t* bytes) {
    if (bytes == nullptr) return FGQA_ERR_INVALID_ARGUMENT;
    int st = plan::validate_paged(a);
    if (st != FGQA_OK) return st;
    DecodePlan plan;
    st = plan::plan_paged(a, &plan);
    if (st != FGQA_OK) return st;
    *bytes = plan.ws_bytes;
    return FGQA_OK;
}

extern "C" int fgqa_decode_paged(const fgqa_decode_paged_args* a, void* stream) {
    int st = plan::validate_paged(a);
    if (st != FGQA_OK) return st;
    st = plan::validate_paged_pointers(a);
    if (st != FGQA_OK) return st;
    if (a->batch == 0) return FGQA_OK;
    DecodePlan plan;
    st = plan::plan_paged(a, &plan);
    if (st != FGQA_OK) return st;

    DecodeParams p;
    p.q = static_cast<const __bf16*>(a->q);
    p.k = static_cast<const __bf16*>(a->k_cache);
    p.v = static_cast<const __bf16*>(a->v_cache);
    p.o = static_cast<__bf16*>(a->o);
    p.lse = a->lse;
    p.seqlens = a->seqlens;
    p.part_o = nullptr;
    p.part_ml = nullptr;
    p.work = nullptr;
    p.prefix = nullptr;
    p.teams = 0;
    p.q_sb = a->q_stride[0];
    p.q_sh = a->q_stride[1];
    p.k_sb = a->k_stride[0];
    p.k_ss = a->k_stride[1];
    p.k_sh = a->k_stride[2];
    p.v_sb = a->v_stride[0];
    p.v_ss = a->v_stride[1];
    p.v_sh = a->v_stride[2];
    p.o_sb = a->o_stride[0];
    p.o_sh = a->o_stride[1];
    p.batch = a->batch;
    p.max_seqlen = a->max_seqlen;
    p.hq = a->num_q_heads;
    p.hkv = a->num_kv_heads;
    p.group = a->num_q_heads / a->num_kv_heads;
    p.nsplit = plan.nsplit;
    p.chunk = plan.chunk;
    p.scale_log2 = a->scale * a->k_scale * kLog2e;
    p.block_table = a->block_table;
    p.bt_stride = a->block_table_stride;
    int shift = 0;
    while ((1 << shift) < a->page_size) ++shift;
    p.page_shift = shift;
    p.num_pages = a->num_pages;
    p.v_scale = a->v_scale;

    const hipStream_t s = static_cast<hipStream_t>(stream);
    int32_t* work = nullptr;
    std::unique_lock<std::mutex> ws_lock;   // held through the launches when the library's buffer is used
    if (plan.ws_bytes > 0) {
        void* ws = a->workspace;
        st = take_workspace(&plan, a->workspace_bytes, s, &ws_lock, &ws);
        if (st != FGQA_OK) return st;
        work = carve_workspace(plan, ws, &p);
    }

    if (a->max_seqlen == 0) {
        launch_combine<false>(p, 1, s);
    } else {
        const int cus = device_cu_count();
        if (cus <= 0) return FGQA_ERR_HIP;
        // Pages of at least one load instruction's rows (4 bf16, 8 fp8) whose
        // bytes stay below 2^31: page segments of min(page, 32) rows, each
        // read through one buffer resource (at BASELINE config 3's lengths
        // with 16- and 64-token pages: bf16 -4 %, fp8 with head pairs -1 to
        // -2 % against the per-row form).
        const bool fp8 = a->kv_dtype == FGQA_KV_FP8_E4M3;
        const bool small_pages = (int64_t)a->page_size * a->k_stride[1] * 2 < ((int64_t)1 << 31) &&
                                 (int64_t)a->page_size * a->v_stride[1] * 2 < ((int64_t)1 << 31);
        const int seg = !small_pages ? 0 : a->page_size >= 32 ? 32 : a->page_size >= 4 ? a->page_size : 0;
        auto pass1 = [&] {
            if (fp8) {
                switch (seg >= 8 ? seg : 0) {
                    case 32: launch_list<kKvPagedFp8, 32>(p, plan.nsplit, cus, s); break;
                    case 16: launch_list<kKvPagedFp8, 16>(p, plan.nsplit, cus, s); break;
                    case 8: launch_list<kKvPagedFp8, 8>(p, plan.nsplit, cus, s); break;
                    default: launch_list<kKvPagedFp8, 0>(p, plan.nsplit, cus, s); break;
                }
            } else {
                switch (seg) {
                    case 32: launch_list<kKvPagedBf16, 32>(p, plan.nsplit, cus, s); break;
                    case 16: launch_list<kKvPagedBf16, 16>(p, plan.nsplit, cus, s); break;
                    case 8: launch_list<kKvPagedBf16, 8>(p, plan.nsplit, cus, s); break;
                    case 4: launch_list<kKvPagedBf16, 4>(p, plan.nsplit, cus, s); break;
                    default: launch_list<kKvPagedBf16, 0>(p, plan.nsplit, cus, s); break;
                }
            }
        };
        run_ragged(p, work, pass1, s);
    }
    if (hipGetLastError() != hipSuccess) return FGQA_ERR_HIP;
    return FGQA_OK;
}
