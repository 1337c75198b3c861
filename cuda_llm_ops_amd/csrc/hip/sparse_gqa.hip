// Sparse-index GQA prefill forward for gfx950.
//
// Stands in for the reference's Triton-only flash_sgqa_forward_bf16_kernel
// (src/python/Triton/SparseGQA/flash_sgqa_kernel.py:15-137).  Query row i of
// head h attends the keys listed in idx[b][h / G][i][0 .. nsparse): an entry is
// used when 0 <= j < Skv and, if causal, j <= i (:98-102); a key listed twice
// counts twice.  Same maths as the dense prefill: fp32 scores, online softmax,
// P rounded to bf16 before P.V with the row sum kept from the fp32 P
// (:110-121), O /= rowsum and lse = max + log(rowsum), or O = 0 and
// lse = -inf for a row with no usable entry (:123-125).
//
// One wave owns one work item: a query position, a KV head and up to 16 of
// its query heads, which share the position's index list.  The heads are the
// N dimension of v_mfma_f32_16x16x32_bf16; per 32-entry step:
//   S^T (32 keys x 16 heads) = K_gathered . Q^T     8 MFMAs, K transposed within
//                                                    lane quads in registers
//   O^T (128 x 16)          += V^T . P^T            8 MFMAs, V read transposed
//                                                    from the wave's LDS tile
//                                                    (ds_read_b64_tr_b16)
// The next step's K and V rows are in flight while a step is computed.
//
// What bounds it: each step gathers 16 KB of K/V rows and does little with
// them.  (Kernel times on one set of lists, repeated; calls on alternating inputs
// take some 10 us more.)  At S = 16384, 512 entries (4.3 GB of gathers) the gathers alone take
// 129 us when they all hit L1, the steps without gathers 112 us; together 155 us
// from L1 and 189 us from the real lists (L2 misses; 4 MB of L2 per XCD against
// 8 MB of K/V).  Before, K went through LDS as well (32 KB of LDS traffic per
// step was the bound: 150 us without any gather) at two waves per SIMD, and
// every list was sorted (37 us): 224 us.  Three waves per SIMD: 165 VGPRs, 11.3
// KB of LDS.  Other forms for small grids and for many keys: SpForm below.
#include <limits.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "fgqa_device.h"
#include "fgqa_internal.h"

namespace fgqa {

struct SparseParams {
    const __bf16* q;
    const __bf16* k;
    const __bf16* v;
    __bf16* o;
    float* lse;
    const int32_t* idx;
    int64_t q_sb, q_ss, q_sh;
    int64_t k_sb, k_ss, k_sh;
    int64_t v_sb, v_ss, v_sh;
    int64_t o_sb, o_ss, o_sh;
    int64_t i_sb, i_sh, i_ss;   // index list strides: batch, kv head, query row
    int batch, sq, skv, hq, hkv, group, nsparse, causal;
    int n_hg;                   // ceil(group / 16) head groups per position
    int64_t n_items;            // batch * hkv * sq * n_hg
    int n_windows, window_shift;   // key windows a list is ordered by, 2^window_shift keys each
    int sorted;                    // kSpFar: ordered by key instead
    FastDiv div_hg, div_sq, div_hkv;
    float scale_log2;           // |scale| * log2(e)
    uint32_t q_sign;            // 0x80008000 when scale < 0 (Q is negated on load)
};

constexpr int kSpWaves = 4;                  // waves (= work items) per workgroup
constexpr int kSpStep = 32;                  // index entries per step
constexpr int kSpRow = 288;                  // V row stride in LDS (256 + 32 bytes)
constexpr int kSpTileBytes = kSpStep * kSpRow;
constexpr int kSpList = 512;                 // index entries taken (and ordered) at a time
constexpr int kSpWaveBytes = kSpTileBytes + kSpList * 4 + 16;   // 11.3 KB of LDS per wave (and a word to drop entries in)
constexpr float kSpMaxP = 65536.f;           // a lane's P of one step, before the max moves

// Lists are taken window by window of keys where K/V outgrow an XCD's L2: all
// waves of the XCD then walk the keys of their prefixes from low to high at
// about the same pace, and a row one wave fetches is often still in L2 when
// another needs it.  Windows of 2048 keys (1 MB of K/V; S = 16384, 512 entries:
// 189 us against 194 with 4096 keys, 193 with 1024, 221 without windows, 202
// fully sorted), but none for fewer than 32 of a list's entries (a window costs
// ~60 instructions: S = 24576, 64 entries 104 us with 12 windows, 90 with 2).
// Up to 8192 keys all K/V fit: one window.
constexpr int kSpWindowLog2 = 11;
constexpr int kSpNoWindows = 8192;
// The kernel's forms.
//  - kSpThree: three waves per SIMD (165 registers), a step of rows in flight.
//  - kSpChain: two waves; a wave's next K rows are gathered before its scores
//    instead of after them (188 registers).  For grids that fit the chip at two
//    workgroups per CU, where a launch is one wave's chain of steps: S = 546,
//    512 entries 19.2 against 21.3 us, S = 2048, 512 entries 29.2 against 31.1;
//    at S = 3000 (750 workgroups) 15.3 against 14.6.
//  - kSpFar: two waves, two steps of rows in flight (249 registers).  For rows
//    that see more than 16384 keys on average (half of them under the causal
//    mask), where L2 serves fewer waves better, and lists of 256 entries or
//    more.  us, three waves / far: 24576 keys, full, 256 entries 291 / 272, 1024
//    entries 813 / 675; 32768 keys, full, 512 entries 634 / 556; 40000 keys,
//    causal, 512 entries 624 / 613; but 24576 keys, causal, 512 entries 316 /
//    337, and 40000 keys, full, 64 entries 196 / 203.
enum SpForm { kSpThree, kSpChain, kSpFar };
constexpr int kSpFarKeys = 16384;
constexpr int kSpFarList = 256;
// kSpFar takes lists of 257 to 512 entries in full key order instead of by
// windows: 65536 keys, 512 entries 1628 against 1635 us (full) and 1179 against
// 1208 (causal), 40000 keys, full 771 against 801; but 256 entries at 24576 keys
// 288 against 274, and 1024 entries (two parts) at 65536 keys 3354 against 3298.
constexpr int kSpSortMin = 257;

// Gathers read whole rows per instruction, in pieces of a quad (K, 64 bytes) or
// of 16 lanes (V, 256 bytes); both run at the same rate (129-132 us for 4.3 GB
// from L1), while a lane-per-row gather makes the L1 handle one access per lane
// and is several times slower.  A 288-byte row stride (256 + 32) keeps both LDS
// patterns of V free of bank conflicts (the b128 writes of one row's 16 chunks,
// and the transposed reads of rows 0..7 x chunks {2dt, 2dt + 1} per 32 lanes).

// Block -> first work item: the last positions first.  Blocks go round-robin
// over the 8 XCDs, so every XCD works through the same positions at the same
// time: each L2 holds rows of the same causal prefix and the XCDs finish
// together.  (Handing each XCD one contiguous range of positions gives the
// XCDs with early positions a prefix that fits their L2 and the others one that
// does not; at S = 32768 the late XCDs then ran 30 % longer per item and the
// launch took 16 % longer.)  Early positions have the fewest usable entries, so
// running them last shortens the tail.
__device__ __forceinline__ int64_t sp_block_first_item(int64_t nblocks) {
    return (nblocks - 1 - (int64_t)blockIdx.x) * kSpWaves;
}

// Lanes 4a .. 4a+3 hold, in r[i], dword c of chunk j of row i (lane 4a + j);
// afterwards lane 4a + j holds chunk i of row j in r[i].  Two dwords (a and b) at
// a time: each of the 16 moves takes the neighbour's register through DPP and
// keeps or replaces by a lane mask (v_cndmask with a DPP source; the masks go
// through vcc).  A DPP read needs two wait states after a VALU write of its
// register: the first s_nop covers what comes before, the order of the moves the
// rest.  The last one keeps an MFMA that follows two states behind the moves (the
// compiler counts no wait states around inline asm).
__device__ __forceinline__ void sp_transpose_quad(uint32_t& a0, uint32_t& a1, uint32_t& a2, uint32_t& a3,
                                                  uint32_t& b0, uint32_t& b1, uint32_t& b2, uint32_t& b3,
                                                  uint64_t bit0, uint64_t bit1) {
    uint32_t t0, t1, t2, t3, u0, u1, u2, u3;
    asm("s_not_b64 vcc, %[m0]\n\t"
        "s_nop 1\n\t"
        "v_cndmask_b32_dpp %[t0], %[a1], %[a0], vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_cndmask_b32_dpp %[t2], %[a3], %[a2], vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_cndmask_b32_dpp %[u0], %[b1], %[b0], vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_cndmask_b32_dpp %[u2], %[b3], %[b2], vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "s_mov_b64 vcc, %[m0]\n\t"
        "v_cndmask_b32_dpp %[t1], %[a0], %[a1], vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_cndmask_b32_dpp %[t3], %[a2], %[a3], vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_cndmask_b32_dpp %[u1], %[b0], %[b1], vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_cndmask_b32_dpp %[u3], %[b2], %[b3], vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "s_not_b64 vcc, %[m1]\n\t"
        "v_cndmask_b32_dpp %[a0], %[t2], %[t0], vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_cndmask_b32_dpp %[a1], %[t3], %[t1], vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_cndmask_b32_dpp %[b0], %[u2], %[u0], vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_cndmask_b32_dpp %[b1], %[u3], %[u1], vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "s_mov_b64 vcc, %[m1]\n\t"
        "v_cndmask_b32_dpp %[a2], %[t0], %[t2], vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_cndmask_b32_dpp %[a3], %[t1], %[t3], vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_cndmask_b32_dpp %[b2], %[u0], %[u2], vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_cndmask_b32_dpp %[b3], %[u1], %[u3], vcc quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1"
        : [a0] "+v"(a0), [a1] "+v"(a1), [a2] "+v"(a2), [a3] "+v"(a3), [b0] "+v"(b0), [b1] "+v"(b1), [b2] "+v"(b2),
          [b3] "+v"(b3), [t0] "=&v"(t0), [t1] "=&v"(t1), [t2] "=&v"(t2), [t3] "=&v"(t3), [u0] "=&v"(u0),
          [u1] "=&v"(u1), [u2] "=&v"(u2), [u3] "=&v"(u3)
        : [m0] "s"(bit0), [m1] "s"(bit1)
        : "vcc", "scc");
}

// The value of lane ^ d: DPP quad permutes for d = 1, 2, a bit-mode swizzle
// inside each half-wave for 4 <= d <= 16, the half-wave swap for 32.
__device__ __forceinline__ int sp_xor(int v, int d, int lane) {
    switch (d) {
        case 1: return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
        case 2: return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, false);   // quad_perm [2,3,0,1]
        case 4: return __builtin_amdgcn_ds_swizzle(v, (4 << 10) | 0x1F);
        case 8: return __builtin_amdgcn_ds_swizzle(v, (8 << 10) | 0x1F);
        case 16: return __builtin_amdgcn_ds_swizzle(v, (16 << 10) | 0x1F);
        default: {
            const auto r = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
            return (int)(lane < 32 ? r[1] : r[0]);
        }
    }
}

// Ascending bitonic sort of a wave's 512 ints, value 8*lane + r in x[r]:
// distances of 8 values or more pair registers across lanes, smaller ones
// pair registers of a lane.  Deterministic (no atomics).
__device__ __forceinline__ void sp_sort512(int (&x)[8], int lane) {
#pragma unroll
    for (int k = 2; k <= 512; k <<= 1)
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
            if (j >= 8) {
                // value e pairs with e ^ j: same register of lane ^ (j / 8);
                // the block of size k holding e sorts up when (e & k) == 0
                const int d = j >> 3;
                const bool keep_min = ((lane & d) == 0) == ((lane & (k >> 3)) == 0);
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    const int o = sp_xor(x[r], d, lane);
                    x[r] = keep_min ? min(x[r], o) : max(x[r], o);
                }
            } else {
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    if (r & j) continue;
                    const bool up = ((8 * lane + r) & k) == 0;
                    const int lo = min(x[r], x[r | j]), hi = max(x[r], x[r | j]);
                    x[r] = up ? lo : hi;
                    x[r | j] = up ? hi : lo;
                }
            }
        }
}

// kSameRows: K and V rows are the same number of bytes apart, so one offset
// (kept in the list instead of the key) addresses both.
template <bool kSameRows, SpForm kForm>
__global__ __launch_bounds__(kSpWaves * kWave, kForm == kSpThree ? 3 : 2) void sparse_prefill_kernel(SparseParams p) {
    __shared__ __attribute__((aligned(16))) unsigned char smem[kSpWaves * kSpWaveBytes];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int64_t item = sp_block_first_item(gridDim.x) + wave;
    if (item >= p.n_items) return;   // the kernel has no barrier: a finished wave may leave
    unsigned char* tile = smem + wave * kSpWaveBytes;   // a step's V rows
    int* il = reinterpret_cast<int*>(tile + kSpTileBytes);

    // (the divisions run on the VALU: readfirstlane tells the compiler the
    // results are wave-uniform, so buffer descriptors stay in SGPRs)
    int hg, pos, kvh, b;
    if (p.n_items < ((int64_t)1 << 31)) {
        const int r0 = fast_div((int)item, p.div_hg), r1 = fast_div(r0, p.div_sq), r2 = fast_div(r1, p.div_hkv);
        hg = (int)item - r0 * p.n_hg;
        pos = r0 - r1 * p.sq;
        kvh = r1 - r2 * p.hkv;
        b = r2;
    } else {
        int64_t rest = item;
        hg = (int)(rest % p.n_hg);
        rest /= p.n_hg;
        pos = (int)(rest % p.sq);
        rest /= p.sq;
        kvh = (int)(rest % p.hkv);
        b = (int)(rest / p.hkv);
    }
    hg = __builtin_amdgcn_readfirstlane(hg);
    pos = __builtin_amdgcn_readfirstlane(pos);
    kvh = __builtin_amdgcn_readfirstlane(kvh);
    b = __builtin_amdgcn_readfirstlane(b);

    const int l16 = lane & 15;
    const int g = lane >> 4;          // 16-lane group
    const int h0 = kvh * p.group + hg * 16;
    const int nh = min(16, p.group - hg * 16);   // real heads in this item

    // Q^T as the B operand: lane (head l16, group g) holds dims 32g + 8ks .. +7
    // of k-step ks, as the K operand below.
    bf16x8_t qop[4];
    {
        const __amdgpu_buffer_rsrc_t qrs =
            make_rsrc(p.q + b * p.q_sb + (int64_t)pos * p.q_ss + (int64_t)h0 * p.q_sh,
                      (uint32_t)((int64_t)(nh - 1) * p.q_sh * 2 + 256));
        const uint32_t qoff = (uint32_t)((int64_t)min(l16, nh - 1) * p.q_sh * 2) + g * 64;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            u32x4_t t = buf_load16(qrs, qoff + ks * 16);
            t = (l16 < nh) ? (t ^ p.q_sign) : u32x4_t{0u, 0u, 0u, 0u};
            qop[ks] = as_bf16x8(t);
        }
    }

    // The index list (entries past nsparse read as 0 and are masked below).
    const __amdgpu_buffer_rsrc_t irs =
        make_rsrc(p.idx + b * p.i_sb + kvh * p.i_sh + (int64_t)pos * p.i_ss, (uint32_t)p.nsparse * 4);
    // K/V rows of this (batch, kv head); rows are addressed by 32-bit offsets.
    // (Skv = 0: empty ranges, every load returns 0 and every entry is masked.
    // The select would otherwise put the descriptors in VGPRs.)
    const uint32_t kss = (uint32_t)(p.k_ss * 2);
    const uint32_t vss = (uint32_t)(p.v_ss * 2);
    const uint32_t kv_rows = (uint32_t)p.skv;
    const uint32_t k_bytes = __builtin_amdgcn_readfirstlane(kv_rows ? (kv_rows - 1) * kss + 256 : 0u);
    const uint32_t v_bytes = __builtin_amdgcn_readfirstlane(kv_rows ? (kv_rows - 1) * vss + 256 : 0u);
    const __amdgpu_buffer_rsrc_t krs = make_rsrc(p.k + b * p.k_sb + kvh * p.k_sh, k_bytes);
    const __amdgpu_buffer_rsrc_t vrs = make_rsrc(p.v + b * p.v_sb + kvh * p.v_sh, v_bytes);

    // Row gathers of step t.  K: instruction (tt, i), lane 4a + j of group g
    // reads chunk 4g + j of entry 16tt + 4a + i (a quad reads 64 bytes of one
    // row, the wave four whole rows); the quad's transposition then leaves entry
    // 16tt + l16 in lane l16, the MFMA's A operand with dims 32g + 8ks .. +7 in
    // register ks.  V: instruction i, group g reads entry 8g + i, a row per 16
    // lanes, into the same row of the LDS tile.
    struct Rows {
        u32x4_t k[2][4], v[8];
    };
    auto issue_k = [&](int t, u32x4_t (&kr)[2][4]) {
        const u32x4_t* w = reinterpret_cast<const u32x4_t*>(il + t * kSpStep + (l16 & 12));
        const u32x4_t r0 = w[0], r1 = w[4];
        const uint32_t chunk = (uint32_t)(g * 64 + (lane & 3) * 16);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            kr[0][i] = buf_load16(krs, (kSameRows ? r0[i] : r0[i] * kss) + chunk);
            kr[1][i] = buf_load16(krs, (kSameRows ? r1[i] : r1[i] * kss) + chunk);
        }
    };
    auto issue_v = [&](int t, u32x4_t (&vr)[8]) {
        const u32x4_t* w = reinterpret_cast<const u32x4_t*>(il + t * kSpStep + g * 8);
        const u32x4_t r0 = w[0], r1 = w[1];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t row = i < 4 ? r0[i] : r1[i - 4];
            vr[i] = buf_load16(vrs, (kSameRows ? row : row * vss) + l16 * 16);
        }
    };
    auto transpose = [&](const u32x4_t (&r)[4], u32x4_t (&o)[4], int d) {
        uint32_t a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = r[i][d], b[i] = r[i][d + 1];
        sp_transpose_quad(a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3], 0xAAAAAAAAAAAAAAAAull, 0xCCCCCCCCCCCCCCCCull);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i][d] = a[i], o[i][d + 1] = b[i];
    };
    auto stage_v = [&](const u32x4_t (&vr)[8]) {
#pragma unroll
        for (int i = 0; i < 8; ++i) *reinterpret_cast<u32x4_t*>(tile + (8 * g + i) * kSpRow + l16 * 16) = vr[i];
    };
    // Transposed V reads: lane (l16, g) of half kh supplies entry 16kh + 4g + l16/4,
    // dims 16dt + 4*(l16 % 4) .. +3, i.e. chunk 2dt + (l16/2) % 2, half l16 % 2.
    const unsigned char* vrd = tile + (4 * g + (l16 >> 2)) * kSpRow + ((l16 >> 1) & 1) * 16 + (l16 & 1) * 8;

    const float c = p.scale_log2;
    float m_run = -INFINITY;   // running max (log2 units) of head l16
    float m_use = 0.f;         // m_run, or 0 while m_run is -inf
    float l_run = 0.f;         // this lane's share of head l16's row sum
    f32x4_t oacc[8];
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) oacc[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // S^T C layout: lane (head l16, group g) register r of tile tt = tile row
    // 16tt + 4g + r, the step's entry of that number.
    f32x4_t s[2];
    bf16x8_t pop;
    auto softmax_p = [&]() -> float {
        float psum = 0.f;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float pv = fast_exp2(__builtin_fmaf(s[tt][r], c, -m_use));
                psum += pv;
                pop[tt * 4 + r] = (__bf16)pv;
            }
        return psum;
    };
    for (int c0 = 0; c0 < p.nsparse; c0 += kSpList) {
        // Up to 512 entries, the usable ones first and window by window
        // (a fixed order, by slot modulo 8 and then lane, in a window) or
        // sorted.  The order of the sum changes by rounding only.
        int x[8];
        {
            const u32x4_t a0 = buf_load16(irs, (uint32_t)(c0 + 8 * lane) * 4);
            const u32x4_t a1 = buf_load16(irs, (uint32_t)(c0 + 8 * lane) * 4 + 16);
            const int lim = p.causal ? min(pos + 1, p.skv) : p.skv;
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const int jj = (int)(r < 4 ? a0[r] : a1[r - 4]);
                const bool ok = c0 + 8 * lane + r < p.nsparse && jj >= 0 && jj < lim;
                x[r] = ok ? jj : -1;
            }
        }
        int at[8], n_valid = 0;
#pragma unroll
        for (int r = 0; r < 8; ++r) at[r] = kSpList;   // unusable: dropped
        const bool sorted = kForm == kSpFar && p.sorted;
        if (sorted) {
#pragma unroll
            for (int r = 0; r < 8; ++r) x[r] = x[r] < 0 ? INT_MAX : x[r];
            sp_sort512(x, lane);
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                n_valid += __builtin_popcountll(__builtin_amdgcn_ballot_w64(x[r] != INT_MAX));
                at[r] = x[r] != INT_MAX ? 8 * lane + r : kSpList;
            }
        }
        for (int w = 0; w < (sorted ? 0 : p.n_windows); ++w) {
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const bool in = (x[r] >> p.window_shift) == w;
                const uint64_t m = __builtin_amdgcn_ballot_w64(in);
                const int rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, n_valid));
                at[r] = in ? rank : at[r];
                n_valid += __builtin_popcountll(m);
            }
        }
        if (n_valid == 0) continue;
        // (the last step's unused entries read row 0 and are masked)
        {
            int4* w = reinterpret_cast<int4*>(il + 8 * lane);
            w[0] = w[1] = make_int4(0, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 8; ++r) il[at[r]] = kSameRows ? (int)((uint32_t)x[r] * kss) : x[r];
        const int steps = (n_valid + kSpStep - 1) / kSpStep;
        constexpr int kAhead = kForm == kSpFar ? 2 : 1;   // steps of rows in flight
        auto step = [&](int t, Rows& rows) {
            const bool more = t + kAhead < steps;
            u32x4_t kt[2][4];
            u32x4_t(&ka)[2][4] = kForm == kSpChain ? kt : rows.k;   // (else in place, no registers to spare)
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int d = 0; d < 4; d += 2) transpose(rows.k[tt], ka[tt], d);
            if constexpr (kForm == kSpChain) {
                if (more) issue_k(t + kAhead, rows.k);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
                s[tt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) s[tt] = mfma16(as_bf16x8(ka[tt][ks]), qop[ks], s[tt]);
            }
            if constexpr (kForm != kSpChain) {
                if (more) issue_k(t + kAhead, rows.k);
                __builtin_amdgcn_sched_barrier(0);
            }
            stage_v(rows.v);
            if (more) issue_v(t + kAhead, rows.v);
            const int nv = n_valid - t * kSpStep;
            if (nv < kSpStep) {
#pragma unroll
                for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[tt][r] = 16 * tt + 4 * g + r < nv ? s[tt][r] : -INFINITY;
            }
            // P against the max so far; the max moves only when it must: at the
            // first step, and when a lane's P sums to more than kSpMaxP (bf16's
            // relative precision does not depend on P's size).
            float lt = softmax_p();
            if (__builtin_amdgcn_ballot_w64(m_run == -INFINITY || !(lt <= kSpMaxP)) != 0) {
                float tmax = -INFINITY;
#pragma unroll
                for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) tmax = fmaxf(tmax, s[tt][r]);
                tmax = half_max(xor_max(tmax, 16)) * c;
                const float m_new = fmaxf(m_run, tmax);
                const float m_new_use = (m_new == -INFINITY) ? 0.f : m_new;
                const float alpha = fast_exp2(m_use - m_new_use);
                l_run *= alpha;
#pragma unroll
                for (int dt = 0; dt < 8; ++dt) oacc[dt] *= alpha;
                m_run = m_new;
                m_use = m_new_use;
                lt = softmax_p();
            }
            l_run += lt;
#pragma unroll
            for (int dt = 0; dt < 8; ++dt) {
                const bf16x4_t lo = lds_read_tr16(reinterpret_cast<const __bf16*>(vrd + dt * 32));
                const bf16x4_t hi = lds_read_tr16(reinterpret_cast<const __bf16*>(vrd + 16 * kSpRow + dt * 32));
                oacc[dt] = mfma16(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), pop, oacc[dt]);
            }
        };
        Rows ra;
        issue_k(0, ra.k);
        issue_v(0, ra.v);
        if constexpr (kForm == kSpFar) {
            Rows rb;
            if (steps > 1) {
                issue_k(1, rb.k);
                issue_v(1, rb.v);
            }
            for (int t = 0; t < steps; t += 2) {
                step(t, ra);
                if (t + 1 < steps) step(t + 1, rb);
            }
        } else {
            for (int t = 0; t < steps; ++t) step(t, ra);
        }
    }

    // Row sums over the four lane groups; then O and the LSE of head l16.
    l_run = half_sum(xor_sum(l_run, 16));
    if (l16 < nh) {
        const int h = h0 + l16;
        const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
        __bf16* orow = p.o + b * p.o_sb + (int64_t)pos * p.o_ss + (int64_t)h * p.o_sh;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
            bf16x4_t w;
#pragma unroll
            for (int r = 0; r < 4; ++r) w[r] = (__bf16)(oacc[dt][r] * inv);
            *reinterpret_cast<bf16x4_t*>(orow + 16 * dt + 4 * g) = w;
        }
        if (p.lse != nullptr && g == 0)
            p.lse[((int64_t)b * p.hq + h) * p.sq + pos] = l_run > 0.f ? m_run * kLn2 + logf(l_run) : -INFINITY;
    }
}

static_assert(kSpWaves == plan::kSparseWaves, "waves per sparse workgroup");

}  // namespace fgqa

using namespace fgqa;

extern "C" int fgqa_sparse_prefill_bf16(const fgqa_sparse_prefill_args* a, void* stream) {
    int st = plan::validate_sparse(a);
    if (st != FGQA_OK) return st;
    if (a->batch == 0 || a->seqlen_q == 0) return FGQA_OK;

    SparseParams p;
    p.q = static_cast<const __bf16*>(a->q);
    p.k = static_cast<const __bf16*>(a->k);
    p.v = static_cast<const __bf16*>(a->v);
    p.o = static_cast<__bf16*>(a->o);
    p.lse = a->lse;
    p.idx = a->kv_indices;
    p.q_sb = a->q_stride[0];
    p.q_ss = a->q_stride[1];
    p.q_sh = a->q_stride[2];
    p.k_sb = a->k_stride[0];
    p.k_ss = a->k_stride[1];
    p.k_sh = a->k_stride[2];
    p.v_sb = a->v_stride[0];
    p.v_ss = a->v_stride[1];
    p.v_sh = a->v_stride[2];
    p.o_sb = a->o_stride[0];
    p.o_ss = a->o_stride[1];
    p.o_sh = a->o_stride[2];
    p.i_sb = a->idx_stride[0];
    p.i_sh = a->idx_stride[1];
    p.i_ss = a->idx_stride[2];
    p.batch = a->batch;
    p.sq = a->seqlen_q;
    p.skv = a->seqlen_kv;
    p.hq = a->num_q_heads;
    p.hkv = a->num_kv_heads;
    p.group = a->num_q_heads / a->num_kv_heads;
    p.nsparse = a->num_sparse_kv;
    p.causal = a->causal ? 1 : 0;
    p.n_hg = (int)ceil_div(p.group, 16);
    p.n_items = (int64_t)p.batch * p.hkv * p.sq * p.n_hg;
    p.div_hg = make_fast_div(p.n_hg);
    p.div_sq = make_fast_div(p.sq);
    p.div_hkv = make_fast_div(p.hkv);
    int shift = 31;
    if (p.skv > kSpNoWindows) {
        const int most = std::max(std::min(p.nsparse, kSpList) / kSpStep, 1);
        for (shift = kSpWindowLog2; ((p.skv - 1) >> shift) >= most;) ++shift;
    }
    p.window_shift = shift;
    p.n_windows = p.skv > 0 ? ((p.skv - 1) >> shift) + 1 : 0;
    p.scale_log2 = score_scale(fabsf(a->scale) * kLog2e);
    p.q_sign = (a->scale < 0.f) ? 0x80008000u : 0u;

    const int64_t blocks = ceil_div(p.n_items, kSpWaves);
    if (blocks >= ((int64_t)1 << 31)) return FGQA_ERR_UNSUPPORTED;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const dim3 grid((unsigned)blocks), threads(kSpWaves * kWave);
    const int cus = device_cu_count();
    if (cus <= 0) return FGQA_ERR_HIP;
    const bool few = blocks <= 2 * cus;
    const bool far = !few && p.nsparse >= kSpFarList && (p.causal ? p.skv / 2 : p.skv) > kSpFarKeys;
    p.sorted = p.nsparse >= kSpSortMin && p.nsparse <= kSpList;
    using Kernel = void (*)(SparseParams);
    const Kernel fns[3][2] = {{sparse_prefill_kernel<false, kSpThree>, sparse_prefill_kernel<true, kSpThree>},
                              {sparse_prefill_kernel<false, kSpChain>, sparse_prefill_kernel<true, kSpChain>},
                              {sparse_prefill_kernel<false, kSpFar>, sparse_prefill_kernel<true, kSpFar>}};
    hipLaunchKernelGGL(fns[few ? kSpChain : far ? kSpFar : kSpThree][p.k_ss == p.v_ss], grid, threads, 0, s, p);
    if (hipGetLastError() != hipSuccess) return FGQA_ERR_HIP;
    return FGQA_OK;
}
