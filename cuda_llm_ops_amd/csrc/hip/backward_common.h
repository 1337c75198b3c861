// Definitions shared by the backward's translation units: the kernel parameter
// block, the LDS row layout and the transposed-read addresses.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "fgqa_device.h"

namespace fgqa {

struct BwdParams {
    const __bf16* q;
    const __bf16* k;
    const __bf16* v;
    const __bf16* o;
    const __bf16* dout;
    const float* lse;
    __bf16* dq;
    __bf16* dk;
    __bf16* dv;
    int64_t q_sb, q_ss, q_sh;
    int64_t k_sb, k_ss, k_sh;
    int64_t v_sb, v_ss, v_sh;
    int64_t o_sb, o_ss, o_sh;
    int64_t do_sb, do_ss, do_sh;
    int64_t dq_sb, dq_ss, dq_sh;
    int64_t dk_sb, dk_ss, dk_sh;
    int64_t dv_sb, dv_ss, dv_sh;
    // workspace
    float* rowstat;   // [B*Hq*Sq][2]: -lse*log2(e) and -delta*scale of each query row
    float* dk_part;   // [n_hsplit][B, Hkv, Skv, D] fp32 partial sums (heads split), else null
    float* dv_part;
    int batch, sq, skv, hq, hkv, group, causal;
    int window;       // > 0: sliding window (causal), row i uses keys (i - window, i]
    // key-major (dK/dV) grid
    int hs;           // query heads per workgroup
    int n_hsplit;     // group / hs
    int n_kvblocks;   // ceil(skv / 128)
    int kv_streams;   // n_hsplit * hkv * batch
    int n_qblocks32;  // ceil(sq / 32)
    // query-major (dQ) grid, as the forward's
    int hb;           // heads per 128-row unit
    int n_hgroups;    // group / hb
    int n_qunits;     // ceil(sq / (128 / hb))
    int q_streams;    // n_hgroups * hkv * batch
    float scale;
    float scale_log2;   // scale * log2(e)
};

constexpr int kBwWaves = 4;
constexpr int kBwThreads = kBwWaves * kWave;
constexpr int kBwRowBytes = kHeadDim * 2;             // one Q / dO / K / V row
constexpr int kBwHiRowBytes = 128;                    // dims 128..191 of a 192-wide Q / K row

// Q, dO, K and V rows (256 B) sit in LDS with their 16-byte chunks permuted:
// chunk c of row r goes to slot c ^ bw_swz(r).  bw_swz is a bijection on
// r % 16 (16 consecutive rows read at the same chunk hit 16 different slots:
// conflict-free b128 row reads) whose top two bits are r % 4 (4 consecutive
// rows read over 4 consecutive chunks hit 4 disjoint slot groups:
// conflict-free transposed reads).
__device__ __forceinline__ int bw_swz(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

__device__ __forceinline__ void bw_dma16(uint32_t lds_addr, uint32_t voffset, __amdgpu_buffer_rsrc_t rsrc) {
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 :: "s"(lds_addr), "v"(voffset), "s"(rsrc) : "memory");
}
__device__ __forceinline__ void bw_dma4(uint32_t lds_addr, uint32_t voffset, __amdgpu_buffer_rsrc_t rsrc) {
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dword %1, %2, 0 offen lds"
                 :: "s"(lds_addr), "v"(voffset), "s"(rsrc) : "memory");
}
__device__ __forceinline__ void bw_wait_vmem() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Byte offset, within a block of 16 swizzled 256-byte rows, that lane supplies
// to a transposed read (ds_read_b64_tr_b16) so that the wave receives the
// 32x32x16 MFMA operand  X[k = row][n = 32*cb + l32]  with the k order used
// throughout: slots 0..3 of lane (l32, half g2) = rows 4*g2 + 0..3 (h8 = 0),
// slots 4..7 = rows 8 + 4*g2 + 0..3 (h8 = 1).  Source lane (g2, gq, l16)
// points at row 4*g2 + l16/4 + 8*h8, columns 32*cb + 16*gq + 4*(l16%4) .. +3.
__device__ __forceinline__ int bw_tr_off(int lane, int cb, int h8) {
    const int l16 = lane & 15, gq = (lane >> 4) & 1, g2 = lane >> 5;
    const int r = 4 * g2 + (l16 >> 2) + 8 * h8;
    const int c = 4 * cb + 2 * gq + ((l16 >> 1) & 1);
    return r * kBwRowBytes + ((c ^ bw_swz(r)) << 4) + 8 * (l16 & 1);
}

// MLA (Q/K head dim 192, V/O 128): a 192-wide Q or K row is kept as a
// 256-byte part (dims 0..127, laid out as above) and a 128-byte part (dims
// 128..191) in a separate tile, whose chunk c of row r sits in slot
// c ^ bw_swz_hi(r).  bw_swz_hi is a bijection on (r / 2) % 8: 16 consecutive
// rows read at one chunk fall in 16 different 16-byte bank groups (rows of
// either parity share none, 128-byte rows alternate halves of a 256-byte
// bank line).  Its top bit is (r / 2) % 2: rows r and r + 2 read over 4
// consecutive chunks land in different 4-chunk halves, so the transposed
// reads are conflict-free too.
__device__ __forceinline__ int bw_swz_hi(int r) { return (((r >> 1) & 1) << 2) | ((r >> 2) & 3); }
// bw_tr_off for the 128-byte part (column block cb = 0, 1: dims 128 + 32cb ..)
__device__ __forceinline__ int bw_tr_off_hi(int lane, int cb, int h8) {
    const int l16 = lane & 15, gq = (lane >> 4) & 1, g2 = lane >> 5;
    const int r = 4 * g2 + (l16 >> 2) + 8 * h8;
    const int c = 4 * cb + 2 * gq + ((l16 >> 1) & 1);
    return r * kBwHiRowBytes + ((c ^ bw_swz_hi(r)) << 4) + 8 * (l16 & 1);
}
template <int kDk>
struct BwDims {
    static_assert(kDk == 128 || kDk == 192, "Q/K head dim");
    static constexpr bool kHi = kDk > 128;        // a 128-byte part per row
    static constexpr int kRowBytes = kDk * 2;     // one Q / K row in HBM
    static constexpr int kSteps = kDk / 16;       // MFMA k-steps of S over the Q/K dim
    static constexpr int kDb = kDk / 32;          // 32-column blocks of dQ / dK
};

__device__ __forceinline__ bf16x8_t tr_pair(const unsigned char* base, int off0, int off1) {
    const bf16x4_t lo = lds_read_tr16(reinterpret_cast<const __bf16*>(base + off0));
    const bf16x4_t hi = lds_read_tr16(reinterpret_cast<const __bf16*>(base + off1));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

template <int N, int I = 0, typename F>
__device__ __forceinline__ void bw_static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        bw_static_for<N, I + 1>(f);
    }
}

// The dK/dV pass (flash_gqa_backward_dkdv.hip) over `units` workgroups: swa
// for a sliding window, dk the Q/K head dim (128 or 192), add_mask unless the
// scale is 0.  Returns an fgqa_status.
int launch_dkdv(const BwdParams& p, bool swa, int dk, bool add_mask, unsigned units, hipStream_t s);

}  // namespace fgqa
