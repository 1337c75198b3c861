// dK / dV pass of the GQA prefill backward for gfx950 (the maths and the other
// passes: flash_gqa_backward.hip).
//
// A workgroup owns a 128-key block of one KV head (wave w: keys 32w..32w+31,
// their K/V rows in registers) and loops over (query head of its subset,
// 32-row query block):  S = Q K^T, dP = dO V^T (Q/dO rows from LDS), P and dS
// on the VALU (in place as bf16 A operands), dV += P^T dO, dK += dS^T Q (dO/Q
// read transposed, ds_read_b64_tr_b16).  dK/dV stay in registers (fp32).
//
// What bounds it: dK, dV and the K/V operands of 32 keys leave room for one
// wave per SIMD, so a step takes as long as the one wave takes to issue it:
// beside an MFMA (32 cycles) there are 28 cycles for anything else, of which a
// VALU instruction takes 5, an exp 9, an LDS read 4 to 5 and a scalar
// instruction 8 (measured; the LDS itself serves 128 KB of these reads in
// about 550 cycles).  A step's 32 MFMAs (1,024 cycles; head dim 192: 40) are
// therefore written as a fixed sequence of slots, one MFMA each, with the rest
// of the work dealt out evenly between them:
//   slots 0 .. kS-1      S(t+1), dP(t+1)
//   slots kS .. kSlots-1 dV, dK += step t
//   P/dS of step t+1     half an element per slot, from slot kV0 of step t to
//                        slot kV0 of step t+1
//   operand reads        kRing slots ahead of their MFMA
//   Q/dO(t+3) loads      a few slots of the first half
//   barrier              kTail slots before the end: the remaining MFMAs have
//                        their operands already, and the next step's first
//                        reads go out between them
// Q/dO are in four LDS buffers: step t reads t and t+1 while t+2 (awaited at
// the step's barrier) and t+3 land.  The addresses advance by vector adds; no
// division and no 64-bit product is left in the step.
// At B=1, S=4096, Hq=16, Hkv=1, D=128, causal: 170.6 us with the order left
// to the compiler's interleave (75 scalar instructions per step, 32 copies of S
// and dP out of the accumulation registers), 133.2 us so (kernel trace, in turn
// on one device); matrix cores busy 38 and 52 % of the kernel's cycles.
#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "backward_common.h"
#include "fgqa_device.h"
#include "fgqa_internal.h"

namespace fgqa {

constexpr int kKvKeys = 128;                          // keys per workgroup
constexpr int kKvRows = 32;                           // query rows per step
constexpr int kKvBufs = 4;                            // Q/dO buffers
constexpr int kKvTileBytes = kKvRows * kBwRowBytes;   // 8 KB: Q or dO of one step
constexpr int kKvStatBytes = kKvRows * 8;             // (-lse*log2e, -delta*scale) of 32 rows, a copy per wave
// LDS: Q[4] | dO[4] | stats[4][wave], and with head dim 192 the 128-byte parts of Q[4]
constexpr int kKvDoOff = kKvBufs * kKvTileBytes;
constexpr int kKvStatOff = 2 * kKvBufs * kKvTileBytes;
constexpr int kKvQHiTileBytes = kKvRows * kBwHiRowBytes;   // 4 KB
constexpr int kKvQHiOff = kKvStatOff + kKvBufs * kBwWaves * kKvStatBytes;
template <int kDk>
constexpr int kv_smem_bytes() { return kKvQHiOff + (kDk > 128 ? kKvBufs * kKvQHiTileBytes : 0); }

constexpr int kRing = 8;   // operands read ahead
constexpr int kTail = 5;   // slots after the barrier

// dV / dK += on an accumulator held in AGPRs (inline asm: the compiler would
// otherwise move the 128 or 160 accumulators between the two halves of the
// register file).  The compiler counts no wait states around inline asm: the
// slots keep the VALU writes of an operand more than 2 states ahead, and
// acc_settle comes before the accumulators are read
// (tests/test_dkdv_isa.py checks the built code).
__device__ __forceinline__ void mfma_acc(f32x16_t& acc, bf16x8_t a, bf16x8_t b) {
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
__device__ __forceinline__ void acc_settle(f32x16_t& acc) { asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" : "+a"(acc)); }

// kSwa: sliding window (a separate instantiation, so the causal kernels carry
// none of its work).  kAddMask: the mask enters as an additive -inf on S (any
// nonzero scale); without it (scale 0, where -inf * 0 is not -inf) as a select
// on P.
template <bool kSwa, int kDk, bool kAddMask>
__global__ __launch_bounds__(kBwThreads, 1) void bwd_dkdv_kernel(BwdParams p) {
    using D = BwDims<kDk>;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    constexpr int kS = D::kHi ? 20 : 16;     // S and dP MFMAs of a step
    constexpr int kG = kS;                   // dV and dK MFMAs of a step
    constexpr int kSlots = kS + kG;
    // half-element m of P/dS(t+1) runs in slot kV0 + m: its S and dP are done
    // by then, and its first bf16 operands (m = 4) come after the MFMAs that
    // still read the previous step's
    constexpr int kV0 = kS + kG / 2 - 4;
    static_assert(kSlots % kRing == 0, "ring slots are constants");
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int l32 = lane & 31;
    const int l16 = lane & 15;
    const int g2 = lane >> 5;
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;

    // Block -> (key block, head subset, kv head, batch).  Key blocks in
    // ascending order: under the causal mask block 0 sees every query block,
    // so the heaviest workgroups are dispatched first.
    const int stream = blockIdx.x % p.kv_streams;
    const int kb = blockIdx.x / p.kv_streams;
    const int hsp = stream % p.n_hsplit;
    const int kvh = (stream / p.n_hsplit) % p.hkv;
    const int b = stream / (p.n_hsplit * p.hkv);
    const int kv0 = kb * kKvKeys;
    const int h0 = kvh * p.group + hsp * p.hs;

    // K, V rows of this wave's keys as B operands of S = Q K^T, dP = dO V^T:
    // lane (key l32, half g2), k-step ks holds elements 16ks + 8g2 .. +7.
    // Keys >= skv read as zero.
    const uint32_t kss = (uint32_t)(p.k_ss * 2);
    const uint32_t vss = (uint32_t)(p.v_ss * 2);
    const __amdgpu_buffer_rsrc_t krs =
        make_rsrc(p.k + b * p.k_sb + kvh * p.k_sh, (uint32_t)(p.skv - 1) * kss + D::kRowBytes);
    const __amdgpu_buffer_rsrc_t vrs =
        make_rsrc(p.v + b * p.v_sb + kvh * p.v_sh, (uint32_t)(p.skv - 1) * vss + kBwRowBytes);
    const int key = kv0 + 32 * wave + l32;   // this lane's key (column of S)
    bf16x8_t kop[D::kSteps], vop[8];
#pragma unroll
    for (int ks = 0; ks < D::kSteps; ++ks)
        kop[ks] = as_bf16x8(buf_load16(krs, (uint32_t)key * kss + (16 * ks + 8 * g2) * 2));
#pragma unroll
    for (int ks = 0; ks < 8; ++ks)
        vop[ks] = as_bf16x8(buf_load16(vrs, (uint32_t)key * vss + (16 * ks + 8 * g2) * 2));

    // step t: head h0 + t / per_head, query block qb0 + t % per_head
    const int qb0 = p.causal ? min(kv0 / kKvRows, p.n_qblocks32) : 0;
    // a window ends the key block's rows at its last key + window - 1
    const int qb_end = kSwa ? min(p.n_qblocks32, (kv0 + kKvKeys + p.window - 2) / kKvRows + 1) : p.n_qblocks32;
    const int per_head = max(0, qb_end - qb0);
    const int n_iter = p.hs * per_head;

    // The next step to load: per-lane byte offsets from the head's rows (wave w
    // fetches rows 8w..8w+7 of Q and of dO, and its own copy of the 32 rows'
    // statistics).  Rows >= sq lie past the resources' ends and read as zero;
    // past the last step the resources are empty.
    const uint32_t qss = (uint32_t)(p.q_ss * 2);
    const uint32_t dss = (uint32_t)(p.do_ss * 2);
    int ld_h = h0, ld_left = per_head;
    uint32_t q_vo[2], d_vo[2], qhi_vo = 0, st_vo;
    __amdgpu_buffer_rsrc_t qrs, drs, srs;
    auto ld_head = [&]() {   // the first step of head ld_h
        const bool more = ld_h < h0 + p.hs && per_head > 0;
        const int hh = more ? ld_h : h0;
        qrs = make_rsrc(p.q + b * p.q_sb + hh * p.q_sh, more ? (uint32_t)(p.sq - 1) * qss + D::kRowBytes : 0u);
        drs = make_rsrc(p.dout + b * p.do_sb + hh * p.do_sh, more ? (uint32_t)(p.sq - 1) * dss + kBwRowBytes : 0u);
        srs = make_rsrc(p.rowstat + 2 * (((int64_t)b * p.hq + hh) * p.sq), more ? (uint32_t)p.sq * 8 : 0u);
        const int q0 = qb0 * kKvRows;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int r = 8 * wave + 4 * j + (lane >> 4);
            const int slot = (l16 ^ bw_swz(r)) << 4;
            q_vo[j] = (uint32_t)(q0 + r) * qss + slot;
            d_vo[j] = (uint32_t)(q0 + r) * dss + slot;
        }
        if constexpr (D::kHi) {
            // dims 128..191 of rows 8w..8w+7: lane l fills slot l % 8 of row 8w + l / 8
            const int r = 8 * wave + (lane >> 3);
            qhi_vo = (uint32_t)(q0 + r) * qss + kBwRowBytes + 16 * ((lane & 7) ^ bw_swz_hi(r));
        }
        st_vo = (uint32_t)q0 * 8 + lane * 4;
    };
    constexpr int kDma = D::kHi ? 6 : 5;   // load instructions per wave and step
    // load instruction n of the next step, into buffer bf
    auto ld_one = [&](auto nc, auto bf) {
        constexpr int n = decltype(nc)::value, kB = decltype(bf)::value;
        if constexpr (n < 4) {
            constexpr int j = n / 2;
            const uint32_t dst = lds_base + kB * kKvTileBytes + (8 * wave + 4 * j) * kBwRowBytes;
            if constexpr (n % 2 == 0) bw_dma16(dst, q_vo[j], qrs);
            else bw_dma16(dst + kKvDoOff, d_vo[j], drs);
        } else if constexpr (n == 4) {
            bw_dma4(lds_base + kKvStatOff + (kB * kBwWaves + wave) * kKvStatBytes, st_vo, srs);
        } else {
            bw_dma16(lds_base + kKvQHiOff + kB * kKvQHiTileBytes + 8 * wave * kBwHiRowBytes, qhi_vo, qrs);
        }
    };
    auto ld_advance = [&]() {
        if (--ld_left == 0) {
            ++ld_h;
            ld_left = per_head;
            ld_head();
        } else {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                q_vo[j] += kKvRows * qss;
                d_vo[j] += kKvRows * dss;
            }
            if constexpr (D::kHi) qhi_vo += kKvRows * qss;
            st_vo += kKvRows * 8;
        }
    };

    f32x16_t dk_acc[D::kDb], dv_acc[4];
#pragma unroll
    for (int db = 0; db < D::kDb; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) dk_acc[db][i] = 0.f;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) dv_acc[db][i] = 0.f;

    // transposed-read offsets into the Q / dO tiles
    int trq[4][2], trq_hi[2][2];
#pragma unroll
    for (int db = 0; db < 4; ++db) {
        trq[db][0] = bw_tr_off(lane, db, 0);
        trq[db][1] = bw_tr_off(lane, db, 1);
    }
    // b128 row-read offsets of the A operands of S and dP (row l32, chunk 2ks + g2)
    int roff[8], roff_hi[4];
    const int fl = bw_swz(l32);
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) roff[ks] = l32 * kBwRowBytes + (((2 * ks + g2) ^ fl) << 4);
    // (the 128-byte parts and the statistics lie past the 64 KB that an LDS
    // instruction's offset reaches: their areas' starts are in the registers)
    if constexpr (D::kHi) {
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
            trq_hi[cb][0] = kKvQHiOff + bw_tr_off_hi(lane, cb, 0);
            trq_hi[cb][1] = kKvQHiOff + bw_tr_off_hi(lane, cb, 1);
        }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
            roff_hi[ks] = kKvQHiOff + l32 * kBwHiRowBytes + (((2 * ks + g2) ^ bw_swz_hi(l32)) << 4);
    }
    const int soff = kKvStatOff + wave * kKvStatBytes + 4 * g2 * 8;
    const float c2 = p.scale_log2;
    const float scale = p.scale;

    // S = Q K^T and dP = dO V^T of a step: C[q][key], lane (key l32, half g2),
    // register 4i + r <-> query row 8i + 4g2 + r.
    // Element (i, r) of a step's S block is query row q0 + 8i + 4g2 + r; it is
    // masked (P = 0) when 8i + r < m, with m = key - q0 - 4g2 under the causal
    // mask, and (window) when 8i + r > mx, mx = key + window - 1 - q0 - 4g2.
    // Rows >= sq need no mask: their dO rows and -delta*scale read as zero, so
    // P.dO and dS vanish; keys >= skv only reach their own dK/dV rows, which
    // are never stored.
    //
    // kAddMask: the accumulator of a step's S starts at 0 or, on a step whose
    // block the mask cuts (wave-uniform: the diagonal, the window's edge), at
    // ninf for each masked element, ninf = -inf times the sign of scale, so
    // that S * scale * log2(e) is -inf and P = exp2(-inf) = +0 and dS = 0 * x,
    // the values the select gives (for finite Q and K).  Only the first MFMA
    // of S's chain differs between the two.
    const int wk0 = kv0 + 32 * wave;   // the wave's first key
    const int cut_lo = p.causal ? wk0 + 31 : INT32_MIN;          // q0 below it: cut by the causal mask
    const int cut_hi = kSwa ? wk0 + p.window - 32 : INT32_MAX;   // q0 above it: cut by the window
    const float ninf = c2 > 0.f ? -INFINITY : INFINITY;
    auto row_lo = [&](int q0s) { return p.causal ? key - q0s - 4 * g2 : -64; };
    auto row_hi = [&](int q0s) { return key + p.window - 1 - q0s - 4 * g2; };
    auto s_first = [&](const bf16x8_t& a, int q0s) -> f32x16_t {
        f32x16_t z;
#pragma unroll
        for (int i = 0; i < 16; ++i) z[i] = 0.f;
        if (kAddMask && (q0s < cut_lo || (kSwa && q0s > cut_hi))) {
            const int m = row_lo(q0s), mx = row_hi(q0s);
            f32x16_t bias;
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const bool vis = kSwa ? (8 * i + r >= m && 8 * i + r <= mx) : (8 * i + r >= m);
                    bias[4 * i + r] = vis ? 0.f : ninf;
                }
            return mfma32(a, kop[0], bias);
        }
        return mfma32(a, kop[0], z);
    };

    // Operand of slot i (S/dP of the step in buffer BN, dV/dK of the one in BC).
    // S (even) and dP (odd) alternate, then S's k-steps over the 128-byte
    // parts; dV and dK: per 16 rows ks, the column blocks of dV and dK in turn.
    auto fetch = [&](auto ic, auto bc, auto bn) -> bf16x8_t {
        constexpr int i = decltype(ic)::value, BC = decltype(bc)::value, BN = decltype(bn)::value;
        if constexpr (i < 16) {
            return *reinterpret_cast<const bf16x8_t*>(smem + (i % 2 == 0 ? 0 : kKvDoOff) + BN * kKvTileBytes + roff[i / 2]);
        } else if constexpr (i < kS) {
            return *reinterpret_cast<const bf16x8_t*>(smem + BN * kKvQHiTileBytes + roff_hi[(i - 16) % 4]);
        } else {
            constexpr int ks = (i - kS) / (kG / 2), r = (i - kS) % (kG / 2);
            if constexpr (r < 8) {
                const unsigned char* t =
                    smem + (r % 2 == 0 ? kKvDoOff : 0) + BC * kKvTileBytes + ks * 16 * kBwRowBytes;
                return tr_pair(t, trq[(r / 2) % 4][0], trq[(r / 2) % 4][1]);
            } else {
                const unsigned char* t = smem + BC * kKvQHiTileBytes + ks * 16 * kBwHiRowBytes;
                return tr_pair(t, trq_hi[r % 2][0], trq_hi[r % 2][1]);
            }
        }
    };

    // P = exp2(S*scale*log2e - lse*log2e), dS = P (dP - delta) scale, both as
    // bf16 A operands (k-step ks = registers 8ks .. 8ks+7), half an element per
    // call: m = 2e is P of element e, m = 2e + 1 its dS, and the pair (e - 2,
    // e - 1) is rounded at m = 2e for even e.  The statistics of rows 8i .. 8i+7
    // are read at m = 8i - 4 and 8i - 3.
    u32x4_t pop[2], dsop[2];
    f32x4_t st[2][2];
    float pv[4], ds[4];
    [[maybe_unused]] int m_sel = 0, mx_sel = 0;   // the select's bounds (!kAddMask)
    auto softmax = [&](auto mc, const f32x16_t& s, const f32x16_t& dp, auto bi) {
        constexpr int m = decltype(mc)::value, kB = decltype(bi)::value;
        constexpr int mr = m + 4;   // >= 0
        if constexpr (mr % 8 < 2 && mr / 8 < 4)
            st[(mr / 8) & 1][mr % 8] = *reinterpret_cast<const f32x4_t*>(
                smem + kB * kBwWaves * kKvStatBytes + 64 * (mr / 8) + 16 * (mr % 8) + soff);
        if constexpr (m >= 4 && m % 4 == 0) {
            constexpr int e = m / 2 - 2;   // the pair (e, e + 1)
            const bf16x2_t pw = {(__bf16)pv[e & 3], (__bf16)pv[(e & 3) + 1]};
            const bf16x2_t dw = {(__bf16)ds[e & 3], (__bf16)ds[(e & 3) + 1]};
            uint32_t pu = __builtin_bit_cast(uint32_t, pw), du = __builtin_bit_cast(uint32_t, dw);
            asm volatile("" : "+v"(pu), "+v"(du));   // here, not sunk to their MFMA
            pop[e / 8][(e / 2) % 4] = pu;
            dsop[e / 8][(e / 2) % 4] = du;
        }
        if constexpr (m >= 0 && m < 32) {
            constexpr int e = m / 2, i = e / 4, r = e % 4;
            const f32x4_t& w = st[i & 1][r / 2];
            if constexpr (m % 2 == 0) {
                float x = fast_exp2(__builtin_fmaf(s[e], c2, w[2 * (r % 2)]));
                if constexpr (!kAddMask) x = (8 * i + r >= m_sel && (!kSwa || 8 * i + r <= mx_sel)) ? x : 0.f;
                pv[e & 3] = x;
                asm volatile("" : "+v"(pv[e & 3]));   // here, not sunk to its use
            } else {
                ds[e & 3] = pv[e & 3] * __builtin_fmaf(dp[e], scale, w[2 * (r % 2) + 1]);
                asm volatile("" : "+v"(ds[e & 3]));
            }
        }
    };

    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;
    using C2 = std::integral_constant<int, 2>;
    using C3 = std::integral_constant<int, 3>;
    int next_q0 = qb0 * kKvRows;   // first row of the step whose S comes next
    auto advance_q0 = [&]() {
        next_q0 += kKvRows;
        if (next_q0 == qb_end * kKvRows) next_q0 = qb0 * kKvRows;
    };
    bf16x8_t ring[kRing];
    // Step t in buffer BC (= t % 4): sc/dpc hold S/dP(t), sn/dpn receive S/dP(t+1).
    auto step = [&](const f32x16_t& sc, const f32x16_t& dpc, f32x16_t& sn, f32x16_t& dpn, auto bc) {
        constexpr int BC = decltype(bc)::value;
        using BN = std::integral_constant<int, (BC + 1) % 4>;
        using B2 = std::integral_constant<int, (BC + 2) % 4>;
        using BF = std::integral_constant<int, (BC + 3) % 4>;
        [[maybe_unused]] const int q0n = next_q0;
        bw_static_for<kSlots>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const bf16x8_t a = ring[i % kRing];
            if constexpr (i == 0) {
                sn = s_first(a, q0n);
            } else if constexpr (i == 1) {
                f32x16_t z;
#pragma unroll
                for (int x = 0; x < 16; ++x) z[x] = 0.f;
                dpn = mfma32(a, vop[0], z);
            } else if constexpr (i < 16) {
                if constexpr (i % 2 == 0) sn = mfma32(a, kop[i / 2], sn);
                else dpn = mfma32(a, vop[i / 2], dpn);
            } else if constexpr (i < kS) {
                sn = mfma32(a, kop[8 + (i - 16) % 4], sn);
            } else {
                constexpr int ks = (i - kS) / (kG / 2), r = (i - kS) % (kG / 2);
                if constexpr (r < 8 && r % 2 == 0) mfma_acc(dv_acc[r / 2], as_bf16x8(pop[ks]), a);
                else if constexpr (r < 8) mfma_acc(dk_acc[r / 2], as_bf16x8(dsop[ks]), a);
                else mfma_acc(dk_acc[4 + r % 2], as_bf16x8(dsop[ks]), a);
            }
            if constexpr (i + kRing < kSlots) {
                ring[i % kRing] = fetch(std::integral_constant<int, i + kRing>{}, bc, BN{});
            } else if constexpr (i >= kSlots - kTail) {
                if constexpr (i == kSlots - kTail) {
                    // this wave's rows of step t+2 have landed and its reads of
                    // step t's are done; then everyone's
                    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(kDma) : "memory");
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                }
                // the next step's first operands, as ring slots come free
                constexpr int d = i - (kSlots - kTail);
                constexpr int n0 = d < 3 ? 2 * d : d + 3;
                ring[n0] = fetch(std::integral_constant<int, n0>{}, BN{}, B2{});
                if constexpr (d < 3) ring[n0 + 1] = fetch(std::integral_constant<int, n0 + 1>{}, BN{}, B2{});
            }
            if constexpr (i + kSlots - kV0 <= 32) softmax(std::integral_constant<int, i + kSlots - kV0>{}, sc, dpc, bc);
            if constexpr (!kAddMask && i == kV0 - 1) {
                m_sel = row_lo(q0n);
                mx_sel = row_hi(q0n);
            }
            if constexpr (i - kV0 >= -4) softmax(std::integral_constant<int, i - kV0>{}, sn, dpn, BN{});
            if constexpr (i >= 2 && i < 2 + kDma) ld_one(std::integral_constant<int, i - 2>{}, BF{});
            if constexpr (i == 3 + kDma) advance_q0();
            __builtin_amdgcn_sched_barrier(0);
        });
        ld_advance();   // (its branch, like S's first MFMA, at the step's edge)
    };

    f32x16_t sa, dpa, sb, dpb;
    if (n_iter > 0) {
        // steps 0, 1 and 2 into their buffers, 0 and 1 awaited; S/dP(0) and
        // the part of P/dS(0) that a step before it would have run
        ld_head();
        bw_static_for<3>([&](auto bi) {
            bw_static_for<kDma>([&](auto nc) { ld_one(nc, bi); });
            ld_advance();
        });
#pragma unroll
        for (int ks = 0; ks < D::kSteps; ++ks) asm volatile("" : "+a"(kop[ks]));   // K, V live in AGPRs
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) asm volatile("" : "+a"(vop[ks]));
#pragma unroll
        for (int db = 0; db < D::kDb; ++db) asm volatile("" : "+a"(dk_acc[db]));
#pragma unroll
        for (int db = 0; db < 4; ++db) asm volatile("" : "+a"(dv_acc[db]));
        asm volatile("s_waitcnt vmcnt(%0)" :: "n"(kDma) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        m_sel = row_lo(next_q0);
        mx_sel = row_hi(next_q0);
        bw_static_for<kS>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const bf16x8_t a = fetch(ic, C3{}, C0{});
            if constexpr (i == 0) {
                sa = s_first(a, next_q0);
            } else if constexpr (i == 1) {
                f32x16_t z;
#pragma unroll
                for (int x = 0; x < 16; ++x) z[x] = 0.f;
                dpa = mfma32(a, vop[0], z);
            } else if constexpr (i < 16) {
                if constexpr (i % 2 == 0) sa = mfma32(a, kop[i / 2], sa);
                else dpa = mfma32(a, vop[i / 2], dpa);
            } else {
                sa = mfma32(a, kop[8 + (i - 16) % 4], sa);
            }
        });
        advance_q0();
        bw_static_for<kSlots - kV0 + 4>([&](auto ic) {
            softmax(std::integral_constant<int, decltype(ic)::value - 4>{}, sa, dpa, C0{});
        });
        bw_static_for<kRing>([&](auto ic) { ring[decltype(ic)::value] = fetch(ic, C0{}, C1{}); });
        __builtin_amdgcn_sched_barrier(0);
        for (int t = 0;;) {
            step(sa, dpa, sb, dpb, C0{});
            if (++t >= n_iter) break;
            step(sb, dpb, sa, dpa, C1{});
            if (++t >= n_iter) break;
            step(sa, dpa, sb, dpb, C2{});
            if (++t >= n_iter) break;
            step(sb, dpb, sa, dpa, C3{});
            if (++t >= n_iter) break;
        }
#pragma unroll
        for (int db = 0; db < D::kDb; ++db) acc_settle(dk_acc[db]);
#pragma unroll
        for (int db = 0; db < 4; ++db) acc_settle(dv_acc[db]);
    }

    // dK, dV of this wave's keys: C[key][d], lane (d = 32db + l32, half g2),
    // register 4i + r <-> key 32w + 8i + 4g2 + r.  One workgroup per (key
    // block, head subset): bf16 straight out, or an fp32 partial per subset.
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int j = kv0 + 32 * wave + 8 * i + 4 * g2 + r;
            if (j >= p.skv) continue;
            if (p.dk_part != nullptr) {
                const int64_t row = (((int64_t)hsp * p.batch + b) * p.hkv + kvh) * p.skv + j;
                float* dkr = p.dk_part + row * kDk + l32;
                float* dvr = p.dv_part + row * kHeadDim + l32;
#pragma unroll
                for (int db = 0; db < D::kDb; ++db) dkr[32 * db] = dk_acc[db][4 * i + r];
#pragma unroll
                for (int db = 0; db < 4; ++db) dvr[32 * db] = dv_acc[db][4 * i + r];
            } else {
                __bf16* dkr = p.dk + b * p.dk_sb + (int64_t)j * p.dk_ss + kvh * p.dk_sh + l32;
                __bf16* dvr = p.dv + b * p.dv_sb + (int64_t)j * p.dv_ss + kvh * p.dv_sh + l32;
#pragma unroll
                for (int db = 0; db < D::kDb; ++db) dkr[32 * db] = (__bf16)dk_acc[db][4 * i + r];
#pragma unroll
                for (int db = 0; db < 4; ++db) dvr[32 * db] = (__bf16)dv_acc[db][4 * i + r];
            }
        }
}

static_assert(kKvKeys == plan::kBackwardKvKeys, "keys per dK/dV workgroup");

namespace {
template <bool kSwa, int kDk, bool kAddMask>
int launch_one(const BwdParams& p, int slot, unsigned units, hipStream_t s) {
    const int st = set_kernel_smem_once(slot, reinterpret_cast<const void*>(bwd_dkdv_kernel<kSwa, kDk, kAddMask>),
                                        kv_smem_bytes<kDk>());
    if (st != FGQA_OK) return st;
    hipLaunchKernelGGL((bwd_dkdv_kernel<kSwa, kDk, kAddMask>), dim3(units), dim3(kBwThreads), kv_smem_bytes<kDk>(), s,
                       p);
    return FGQA_OK;
}
}  // namespace

int launch_dkdv(const BwdParams& p, bool swa, int dk, bool add_mask, unsigned units, hipStream_t s) {
    // attribute slots 10, 11, 16 and 24..26
    if (dk == 192)
        return add_mask ? launch_one<false, 192, true>(p, 16, units, s) : launch_one<false, 192, false>(p, 26, units, s);
    if (swa)
        return add_mask ? launch_one<true, 128, true>(p, 11, units, s) : launch_one<true, 128, false>(p, 25, units, s);
    return add_mask ? launch_one<false, 128, true>(p, 10, units, s) : launch_one<false, 128, false>(p, 24, units, s);
}

}  // namespace fgqa
