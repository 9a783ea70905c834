// Kernels of the ragged multi-sequence batch (continuous batching), gfx950.
//
// Reference semantics: multi_token_forward (src/model/multi_forward.rs:49-243)
// extended with a pre-filled int8 KV cache, i.e. for every sequence the
// tokens go through forward_with_cache_into one after another
// (src/model/generate.rs:151-160; src/model/cached_forward.rs:164-502).
// Every per-token quantity is computed with the same operations, in the same
// order, as the single-token decode kernels, so a batch is bit-identical to
// that sequence of single-token steps:
//   * the BitLinear dot products are exact integers, here from int8 MFMA
//     (v_mfma_i32_16x16x64_i8) over all tokens at once;
//   * RMSNorm, the int8 quantiser, RoPE, the KV quantiser and attention run
//     per token exactly as in the decode kernels (exact sequential sums).
#include <algorithm>

#include "wm_internal.h"
#include "wm_norm.h"
#include "wm_seqsum.h"

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// I2_S x int8 GEMM on MFMA
// ---------------------------------------------------------------------------
//
// One workgroup = four 64-row groups x 64 tokens: wave w owns group
// 4 * blockIdx.x + w (of whichever tensor it falls in) and all 64 tokens,
// i.e. 4 row tiles x 4 token tiles = 16 MFMAs (v_mfma_i32_16x16x64_i8) per
// 64-column chunk.  MFMA operands, lane l = 16 * seg + r:
//   A (weights): row r of a 16-row tile, dword seg of the row's 16-byte
//                chunk = 16 codes, expanded to one byte each ({0,1,2} =
//                ternary + 1);
//   B (activations): token r of a 16-token tile, the 16 bytes of the same
//                columns (the GEMM activation layout stores them
//                contiguously);
//   D: lane l holds rows 4*seg .. 4*seg+3 of token r.
// Σ_k (t_k + 1)·a_k - Σ_k a_k = Σ_k t_k·a_k is exact in i32 for any k order.
// Activations and weights go through LDS in blocks of kGemmKB chunks, in a
// ring of ST blocks: ST - 1 blocks of direct global->LDS loads are in flight
// while the waves compute the oldest one.  Each activation byte is read
// from L2 once per NG groups, and each B fragment read from LDS feeds four
// MFMAs.  Launches with few workgroups use k_i2s_gemm_kw below instead.
struct gemm_args {
    wm_gemm_desc d[WM_GEMM_MAX_DESC];
    uint32_t group_end[WM_GEMM_MAX_DESC];
    int n_desc;
    uint32_t n_groups;  // over all tensors
    uint32_t n_chunks;
    const uint8_t *act;
    uint32_t m, m_pad;
    const wm_act_meta *meta;
    float *y;
    uint32_t ldy;
};

__device__ __forceinline__ v4i expand_codes(uint32_t w) {
    // byte g of w holds the codes of columns g (bits 7:6), 32+g, 64+g, 96+g
    // of its 32-column quarter block: one shift and mask per quarter.
    const uint32_t m = 0x03030303u;
    v4i a;
    a.x = (int)((w >> 6) & m);
    a.y = (int)((w >> 4) & m);
    a.z = (int)((w >> 2) & m);
    a.w = (int)(w & m);
    return a;
}

constexpr uint32_t kGemmKB = 4;  // chunks per LDS block
constexpr uint32_t kGemmActChunk = WM_GEMM_TILE_TOKENS * 64;  // bytes of a chunk's activation tile
// LDS of a workgroup over NG 64-row groups: a ring of ST blocks of kGemmKB
// chunks (activations, then the groups' weights), later the output tile
template <int NG>
constexpr uint32_t gemm_block_bytes() { return kGemmKB * (kGemmActChunk + NG * 1024u); }
template <int NG>
constexpr uint32_t gemm_out_stride() { return NG * 64u + 4u; }  // floats per token row of the output tile
template <int NG, int ST>
constexpr size_t gemm_lds_bytes() {
    return (size_t)ST * gemm_block_bytes<NG>() > (size_t)WM_GEMM_TILE_TOKENS * gemm_out_stride<NG>() * 4
               ? (size_t)ST * gemm_block_bytes<NG>()
               : (size_t)WM_GEMM_TILE_TOKENS * gemm_out_stride<NG>() * 4;
}

// s_waitcnt vmcnt(N), the other counters left alone (gfx9 encoding: vmcnt
// in bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8)
template <uint32_t N>
__device__ __forceinline__ void gemm_vm_wait() {
    static_assert(N < 64, "vmcnt is six bits");
    __builtin_amdgcn_s_waitcnt((int)((N & 15u) | ((N >> 4) << 14) | (7u << 4) | (15u << 8)));
}
// wait until at most `blocks` blocks of this wave's loads, PER loads each,
// are still in flight (loads complete in issue order)
template <uint32_t PER>
__device__ __forceinline__ void gemm_wait_blocks(uint32_t blocks) {
    if (blocks == 0) gemm_vm_wait<0>();
    else if (blocks == 1) gemm_vm_wait<PER>();
    else if (blocks == 2) gemm_vm_wait<2 * PER>();
    else if (blocks == 3) gemm_vm_wait<3 * PER>();
    else gemm_vm_wait<4 * PER>();
}
constexpr int kGemmMaxStages = 6;  // gemm_wait_blocks covers up to 4 blocks ahead of the one waited for

// 16-byte slot of (token t, segment g) in a chunk's activation tile in LDS:
// the segment is XOR-swizzled by bits 3:2 of the token, so that the 16 lanes
// reading segment g of tokens r..r+15 hit 16 different bank groups.
__device__ __forceinline__ uint32_t gemm_act_slot(uint32_t t, uint32_t g) {
    return t * 4 + (g ^ ((t >> 2) & 3u));
}

struct gemm_group {
    const uint8_t *w;
    uint32_t g, row0, out_dim;
    float scale;
    bool live;
};

__device__ __forceinline__ gemm_group gemm_group_of(const gemm_args &a, uint32_t gid) {
    // the tensor of global group gid, by selects (no dynamic index into the argument block)
    gemm_group r{a.d[0].w, gid, a.d[0].out_row0, a.d[0].out_dim, a.d[0].scale, gid < a.n_groups};
#pragma unroll
    for (int i = 1; i < WM_GEMM_MAX_DESC; i++) {
        const bool in = i < a.n_desc && gid >= a.group_end[i - 1];
        r.w = in ? a.d[i].w : r.w;
        r.g = in ? gid - a.group_end[i - 1] : r.g;
        r.row0 = in ? a.d[i].out_row0 : r.row0;
        r.out_dim = in ? a.d[i].out_dim : r.out_dim;
        r.scale = in ? a.d[i].scale : r.scale;
    }
    return r;
}

// NG 64-row groups per workgroup of four waves: wave w works on group
// w / (4 / NG) and on TPW = NG token tiles of 16 (NG = 4: one group and all
// 64 tokens per wave; NG = 1: the workgroup's one group, 16 tokens per wave).
// ST: blocks in the LDS ring.
template <int NG, int ST>
__global__ __launch_bounds__(256) void k_i2s_gemm(gemm_args a) {
    static_assert(ST >= 2 && ST <= kGemmMaxStages, "ring size");
    constexpr uint32_t WPG = 4 / NG, TPW = 4 / WPG;  // waves per group, token tiles per wave
    constexpr uint32_t kBlock = gemm_block_bytes<NG>(), kWChunk = NG * 1024u;
    constexpr uint32_t kOutStride = gemm_out_stride<NG>();
    extern __shared__ __align__(16) uint8_t gl[];  // [ST] blocks (activations, weights), then the output tile
    const uint32_t tid = threadIdx.x;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6)), lane = tid & 63;
    const uint32_t r16 = lane & 15, seg = lane >> 4;
    const uint32_t q = wave / WPG, s0 = (wave % WPG) * TPW;  // this wave's group and first token tile
    const gemm_group G = gemm_group_of(a, blockIdx.x * NG + q);
    const uint32_t n0 = blockIdx.y * WM_GEMM_TILE_TOKENS;
    const uint32_t c0 = 0, c1 = a.n_chunks;  // the chunks [c0, c1)
    // Both operands reach LDS by direct global->LDS loads (global_load_lds:
    // lane l of a wave writes 16 bytes at the wave's LDS base + 16 l), a
    // block of kGemmKB chunks at a time.  Per chunk:
    //   activations: wave w fills slots 64 w .. 64 w + 63 of the 256-slot
    //     tile; slot p holds token p / 4, segment (p % 4) ^ bits 3:2 of the
    //     token (gemm_act_slot);
    //   weights: wave w < NG copies group w's 1024-byte chunk (row r's 16
    //     bytes to slot r); a group past the last is group 0's copy, its
    //     sums discarded.
    const gemm_group GW = gemm_group_of(a, blockIdx.x * NG + (wave < NG ? wave : 0));
    const uint8_t *wsrc = (GW.live ? GW.w + (uint64_t)GW.g * a.n_chunks * 1024 : a.d[0].w) + lane * 16;
    const uint32_t p_act = wave * 64 + lane, t_act = p_act >> 2;
    const uint32_t g_act = (p_act & 3u) ^ ((t_act >> 2) & 3u);
    const uint8_t *asrc = a.act + (uint64_t)(n0 + t_act) * 64 + g_act * 16;
    const uint64_t cstride = (uint64_t)a.m_pad * 64;
    const uint32_t nblocks = (c1 - c0 + kGemmKB - 1) / kGemmKB;
#define WM_GEMM_ISSUE(BLK, BUF)                                                                  \
    do {                                                                                         \
        uint8_t *blk_ = gl + (BUF) * kBlock;                                                     \
        _Pragma("unroll") for (uint32_t kb = 0; kb < kGemmKB; kb++) {                            \
            /* past the range: its last chunk again, never read */                               \
            const uint32_t c = min(c0 + (BLK) * kGemmKB + kb, c1 - 1);                           \
            __builtin_amdgcn_global_load_lds(asrc + c * cstride,                                 \
                                             blk_ + kb * kGemmActChunk + wave * 1024, 16, 0, 0); \
            if (wave < NG)                                                                       \
                __builtin_amdgcn_global_load_lds(wsrc + (uint64_t)c * 1024,                      \
                                                 blk_ + kGemmKB * kGemmActChunk + kb * kWChunk + \
                                                     wave * 1024, 16, 0, 0);                     \
        }                                                                                        \
    } while (0)
    v4i acc[4][TPW];
#pragma unroll
    for (int rt = 0; rt < 4; rt++)
#pragma unroll
        for (uint32_t s = 0; s < TPW; s++) acc[rt][s] = v4i{0, 0, 0, 0};
    // this lane's B slots (token tile s0 + s: token 16 (s0 + s) + r16,
    // segment seg) and A words (row tile rt: row 16 rt + r16, dword seg)
    uint32_t b_off[TPW];
#pragma unroll
    for (uint32_t s = 0; s < TPW; s++) b_off[s] = gemm_act_slot((s0 + s) * 16 + r16, seg) * 16;
    const uint32_t a_off = kGemmKB * kGemmActChunk + q * 1024 + r16 * 16 + seg * 4;
    // blocks 0 .. ST - 2 in flight before the loop; block b + ST - 1 goes out
    // once every wave has finished block b - 1, whose slot it takes
#pragma unroll
    for (uint32_t b = 0; b + 1 < (uint32_t)ST; b++)
        if (b < nblocks) WM_GEMM_ISSUE(b, b);
    uint32_t slot = 0;  // b % ST
    for (uint32_t b = 0; b < nblocks; b++) {
        // this wave's loads of block b: the blocks issued after it may stay in flight
        const uint32_t ahead = min((uint32_t)ST - 2, nblocks - 1 - b);
        if (wave < NG) gemm_wait_blocks<2 * kGemmKB>(ahead);
        else gemm_wait_blocks<kGemmKB>(ahead);
        // everyone's loads of block b, and block b - 1 fully read.  A bare
        // barrier: __syncthreads()' release fence would wait for every load
        // in flight (vmcnt(0)), the later blocks' included.
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (b + ST - 1 < nblocks) WM_GEMM_ISSUE(b + ST - 1, slot == 0 ? ST - 1 : slot - 1);
        const uint8_t *blk = gl + slot * kBlock;
        slot = slot + 1 == (uint32_t)ST ? 0u : slot + 1;
        const uint32_t kbn = min(kGemmKB, c1 - c0 - b * kGemmKB);
        // The block's fragments first, then its MFMAs.  A chunk past the
        // range (a copy of the last one) gets zero codes, which add nothing:
        // no branch around the MFMAs, so the sums stay in their registers.
        v4i bv[kGemmKB][TPW];
        uint32_t wv[kGemmKB][4];
#pragma unroll
        for (uint32_t kb = 0; kb < kGemmKB; kb++) {
#pragma unroll
            for (uint32_t s = 0; s < TPW; s++)
                bv[kb][s] = *reinterpret_cast<const v4i *>(blk + kb * kGemmActChunk + b_off[s]);
#pragma unroll
            for (int rt = 0; rt < 4; rt++) {
                const uint32_t w = *reinterpret_cast<const uint32_t *>(blk + a_off + kb * kWChunk + rt * 256);
                wv[kb][rt] = kb < kbn ? w : 0u;
            }
        }
#pragma unroll
        for (uint32_t kb = 0; kb < kGemmKB; kb++) {
#pragma unroll
            for (int rt = 0; rt < 4; rt++) {
                const v4i av = expand_codes(wv[kb][rt]);
#pragma unroll
                for (uint32_t s = 0; s < TPW; s++)
                    acc[rt][s] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bv[kb][s], acc[rt][s], 0, 0, 0);
            }
        }
    }
#undef WM_GEMM_ISSUE
    __syncthreads();  // every wave is done with the ring before the output tile reuses it
    // epilogue: y = (w_scale * act_scale) * (dot as f32)   (bitlinear_sse2.rs:327-339),
    // through LDS so that every token's outputs of a group leave as 256
    // contiguous bytes (the MFMA layout gives each lane 4 rows of one token)
    float *ot = reinterpret_cast<float *>(gl);  // [64 tokens][kOutStride]
#pragma unroll
    for (uint32_t s = 0; s < TPW; s++) {
        const uint32_t tl = (s0 + s) * 16 + r16;
        const wm_act_meta mt = a.meta[min(n0 + tl, a.m - 1)];
        const float comb = G.scale * mt.scale;
#pragma unroll
        for (int rt = 0; rt < 4; rt++) {
            float4 o;
            o.x = comb * (float)(acc[rt][s].x - mt.asum);
            o.y = comb * (float)(acc[rt][s].y - mt.asum);
            o.z = comb * (float)(acc[rt][s].z - mt.asum);
            o.w = comb * (float)(acc[rt][s].w - mt.asum);
            *reinterpret_cast<float4 *>(ot + tl * kOutStride + q * 64 + rt * 16 + seg * 4) = o;
        }
    }
    __syncthreads();
    // the 64 x 64 outputs of group g: 1024 float4, four per thread
#pragma unroll
    for (uint32_t g = 0; g < (uint32_t)NG; g++) {
        const gemm_group Q = gemm_group_of(a, blockIdx.x * NG + g);
        if (!Q.live) break;
        const uint32_t base = Q.g * 64;
        const bool vec = ((Q.row0 | a.ldy) & 3u) == 0;
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) {
            const uint32_t idx = tid + k * 256, tl = idx >> 4, c4 = (idx & 15) * 4;
            const uint32_t t = n0 + tl;
            if (t >= a.m) continue;
            const float4 o = *reinterpret_cast<const float4 *>(ot + tl * kOutStride + g * 64 + c4);
            float *dst = a.y + (uint64_t)t * a.ldy + Q.row0 + base + c4;
            if (vec && base + c4 + 4 <= Q.out_dim) {
                *reinterpret_cast<float4 *>(dst) = o;
            } else {
                const float ov[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (base + c4 + r < Q.out_dim) dst[r] = ov[r];
            }
        }
    }
}

// The same GEMM with the K dimension split over the four waves instead of
// the tokens: every wave computes the workgroup's whole NG*64-row x 64-token
// tile over chunks w, w + 4, w + 8, ..., so each code word is expanded once
// per workgroup and feeds 4 MFMAs.  A wave's operands are its own: each
// wave keeps a private ring of ST chunk slots in LDS, filled by direct
// global->LDS loads, and needs no barrier in the K loop.  While the MFMAs of
// chunk j run, chunk j + 1's fragments are read from LDS and chunk j + ST
// is in flight.  The four partial tiles are added through LDS at the end
// (exact: integers).
template <int NG>
constexpr uint32_t gemm_kw_slot_bytes() { return 4096u + NG * 1024u; }  // B tile, then NG groups' codes
template <int NG, int ST>
constexpr size_t gemm_kw_lds_bytes() {
    constexpr size_t ring = (size_t)4 * ST * gemm_kw_slot_bytes<NG>();
    constexpr size_t red = (size_t)4 * 16 * 64 * 16;  // one group's four partial tiles
    constexpr size_t out = (size_t)WM_GEMM_TILE_TOKENS * gemm_out_stride<NG>() * 4;
    return ring > red ? (ring > out ? ring : out) : (red > out ? red : out);
}
template <int NG, int ST>
__global__ __launch_bounds__(256) void k_i2s_gemm_kw(gemm_args a) {
    static_assert(ST >= 2 && ST <= kGemmMaxStages, "ring size");
    constexpr uint32_t kOutStride = gemm_out_stride<NG>();
    constexpr uint32_t kSlot = gemm_kw_slot_bytes<NG>();
    constexpr uint32_t kLoads = 4 + NG;  // global->LDS loads per chunk and wave
    extern __shared__ __align__(16) uint8_t gl[];
    const uint32_t tid = threadIdx.x;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6)), lane = tid & 63;
    const uint32_t r16 = lane & 15, seg = lane >> 4;
    const uint32_t n0 = blockIdx.y * WM_GEMM_TILE_TOKENS;
    const uint32_t nc = a.n_chunks;
    uint8_t *ring = gl + wave * ST * kSlot;
    // Loads, lane l: B tile s: LDS slot l of 16 bytes holds token 16 s + l / 4,
    // segment (l % 4) ^ bits 3:2 of the token (gemm_act_slot, so that the
    // MFMA reads below hit distinct banks); A of group g: row l's 16 bytes.
    const uint32_t t_act = lane >> 2, g_act = (lane & 3u) ^ ((t_act >> 2) & 3u);
    const uint8_t *bsrc = a.act + (uint64_t)(n0 + t_act) * 64 + g_act * 16;
    const uint64_t cstride = (uint64_t)a.m_pad * 64;
    const uint8_t *wsrc[NG];
#pragma unroll
    for (int g = 0; g < NG; g++) {
        const gemm_group Gg = gemm_group_of(a, blockIdx.x * NG + g);
        // a group past the last reads group 0's codes; its sums are discarded
        wsrc[g] = (Gg.live ? Gg.w + (uint64_t)Gg.g * nc * 1024 : a.d[0].w) + lane * 16;
    }
    // this wave's chunk j is wave + 4 j; past the end: the last chunk again
    // (its codes are zeroed before use)
#define WM_KW_ISSUE(J, SLOT)                                                                      \
    do {                                                                                          \
        const uint32_t c_ = min(wave + 4u * (J), nc - 1);                                         \
        uint8_t *d_ = ring + (SLOT) * kSlot;                                                      \
        _Pragma("unroll") for (int s_ = 0; s_ < 4; s_++)                                          \
            __builtin_amdgcn_global_load_lds(bsrc + c_ * cstride + s_ * 1024, d_ + s_ * 1024, 16, 0, 0); \
        /* (the source through a local: an array element passed to the builtin                   \
           makes the host pass drop the kernel's launch stub) */                                  \
        _Pragma("unroll") for (int g_ = 0; g_ < NG; g_++) {                                       \
            const uint8_t *w_ = wsrc[g_] + (uint64_t)c_ * 1024;                                   \
            __builtin_amdgcn_global_load_lds(w_, d_ + 4096 + g_ * 1024, 16, 0, 0);                \
        }                                                                                         \
    } while (0)
    // this lane's fragments in a slot: B of token tile s (token 16 s + r16,
    // segment seg), A of group g, row tile rt (row 16 rt + r16, dword seg)
    const uint32_t b_off = gemm_act_slot(r16, seg) * 16;
    const uint32_t a_off = 4096u + r16 * 16 + seg * 4;
#define WM_KW_READ(SLOT, BV, AV)                                                                  \
    do {                                                                                          \
        const uint8_t *q_ = ring + (SLOT) * kSlot;                                                \
        _Pragma("unroll") for (int s_ = 0; s_ < 4; s_++)                                          \
            BV[s_] = *reinterpret_cast<const v4i *>(q_ + s_ * 1024 + b_off);                      \
        _Pragma("unroll") for (int g_ = 0; g_ < NG; g_++)                                         \
            _Pragma("unroll") for (int rt_ = 0; rt_ < 4; rt_++)                                   \
                AV[g_][rt_] = *reinterpret_cast<const uint32_t *>(q_ + a_off + g_ * 1024 + rt_ * 256); \
    } while (0)
    v4i acc[NG][4][4];
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
        for (int rt = 0; rt < 4; rt++)
#pragma unroll
            for (int s = 0; s < 4; s++) acc[g][rt][s] = v4i{0, 0, 0, 0};
    const uint32_t J = (nc + 3) / 4;  // steps (the waves with fewer chunks zero their last codes)
    // chunks 0 .. ST - 1 in flight, chunk 0 read
#pragma unroll
    for (int u = 0; u < ST; u++)
        if ((uint32_t)u < J) WM_KW_ISSUE((uint32_t)u, (uint32_t)u);
    if (J > 1) gemm_wait_blocks<kLoads>(min((uint32_t)ST - 1, J - 1));
    else gemm_vm_wait<0>();
    // two register sets, used alternately (no copies between steps)
    v4i b0[4], b1[4];
    uint32_t a0[NG][4], a1[NG][4];
    WM_KW_READ(0u, b0, a0);
    uint32_t slot = 0;  // j % ST
#define WM_KW_STEP(JJ, BC, AC, BN, AN)                                                            \
    do {                                                                                          \
        const uint32_t j_ = (JJ);                                                                 \
        const uint32_t nslot_ = slot + 1 == (uint32_t)ST ? 0u : slot + 1;                         \
        /* chunk j + 1 has landed when at most the chunks issued after it are in                 \
           flight: j + 2 .. min(j + ST - 1, J - 1).  Past the last chunk the read                \
           is of a stale slot, never used. */                                                     \
        gemm_wait_blocks<kLoads>(j_ + 1 < J ? min((uint32_t)ST - 2, J - 2 - j_) : 0u);            \
        asm volatile("" ::: "memory");                                                            \
        WM_KW_READ(nslot_, BN, AN);                                                               \
        __builtin_amdgcn_sched_barrier(0); /* the reads go out before this chunk's MFMAs */       \
        const bool live_ = wave + 4u * j_ < nc;                                                   \
        _Pragma("unroll") for (int g = 0; g < NG; g++)                                            \
            _Pragma("unroll") for (int rt = 0; rt < 4; rt++) {                                    \
                const v4i av = expand_codes(live_ ? AC[g][rt] : 0u);                              \
                _Pragma("unroll") for (int s = 0; s < 4; s++)                                     \
                    acc[g][rt][s] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, BC[s], acc[g][rt][s], 0, 0, 0); \
            }                                                                                     \
        /* slot j is free once its fragments are in registers (the MFMAs above                   \
           have them); chunk j + ST takes it.  The wait is for chunk j + 1's reads               \
           too, which had this chunk's MFMAs to land. */                                          \
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                                        \
        if (j_ + ST < J) WM_KW_ISSUE(j_ + ST, slot);                                              \
        slot = nslot_;                                                                            \
    } while (0)
    // an even number of steps: a step past J has zero codes and adds nothing
    // (no branch around the MFMAs, so the sums stay in place)
    for (uint32_t j = 0; j < J; j += 2) {
        WM_KW_STEP(j, b0, a0, b1, a1);
        WM_KW_STEP(j + 1, b1, a1, b0, a0);
    }
#undef WM_KW_STEP
#undef WM_KW_ISSUE
#undef WM_KW_READ
    __syncthreads();  // every wave is done with its ring
    // the four waves' tiles through LDS, one group at a time; wave w then
    // owns row tile w
    v4i *red = reinterpret_cast<v4i *>(gl);  // [4 waves][4 rt][4 s][64 lanes]
    v4i sum[NG][4];
#pragma unroll
    for (int g = 0; g < NG; g++) {
        if (g > 0) __syncthreads();  // the previous group's sums are read
#pragma unroll
        for (int rt = 0; rt < 4; rt++)
#pragma unroll
            for (int s = 0; s < 4; s++) red[((wave * 4 + rt) * 4 + s) * 64 + lane] = acc[g][rt][s];
        __syncthreads();
#pragma unroll
        for (int s = 0; s < 4; s++) {
            v4i t = red[((0 * 4 + wave) * 4 + s) * 64 + lane];
#pragma unroll
            for (uint32_t v = 1; v < 4; v++) t += red[((v * 4 + wave) * 4 + s) * 64 + lane];
            sum[g][s] = t;
        }
    }
    __syncthreads();  // the output tile reuses the reduction area
    // epilogue: y = (w_scale * act_scale) * (dot as f32)   (bitlinear_sse2.rs:327-339)
    float *ot = reinterpret_cast<float *>(gl);  // [64 tokens][kOutStride]
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const uint32_t tl = (uint32_t)s * 16 + r16;
        const wm_act_meta mt = a.meta[min(n0 + tl, a.m - 1)];
#pragma unroll
        for (int g = 0; g < NG; g++) {
            const float comb = gemm_group_of(a, blockIdx.x * NG + g).scale * mt.scale;
            float4 o;
            o.x = comb * (float)(sum[g][s].x - mt.asum);
            o.y = comb * (float)(sum[g][s].y - mt.asum);
            o.z = comb * (float)(sum[g][s].z - mt.asum);
            o.w = comb * (float)(sum[g][s].w - mt.asum);
            *reinterpret_cast<float4 *>(ot + tl * kOutStride + g * 64 + wave * 16 + seg * 4) = o;
        }
    }
    __syncthreads();
    // the 64 x 64 outputs of group g: 1024 float4, four per thread
#pragma unroll
    for (uint32_t g = 0; g < (uint32_t)NG; g++) {
        const gemm_group Q = gemm_group_of(a, blockIdx.x * NG + g);
        if (!Q.live) break;
        const uint32_t base = Q.g * 64;
        const bool vec = ((Q.row0 | a.ldy) & 3u) == 0;
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) {
            const uint32_t idx = tid + k * 256, tl = idx >> 4, c4 = (idx & 15) * 4;
            const uint32_t t = n0 + tl;
            if (t >= a.m) continue;
            const float4 o = *reinterpret_cast<const float4 *>(ot + tl * kOutStride + g * 64 + c4);
            float *dst = a.y + (uint64_t)t * a.ldy + Q.row0 + base + c4;
            if (vec && base + c4 + 4 <= Q.out_dim) {
                *reinterpret_cast<float4 *>(dst) = o;
            } else {
                const float ov[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (base + c4 + r < Q.out_dim) dst[r] = ov[r];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// per-row absmax int8 (bitlinear_sse2.rs:285-304) into the GEMM layout
// ---------------------------------------------------------------------------
// 512 threads per row: two rows per CU (at up to 128 VGPRs a thread), so
// that a batch of up to 512 rows runs in one round over the 256 CUs
constexpr int kRowThreads = 512;

__global__ __launch_bounds__(kRowThreads) void k_quantize_rows(const float *__restrict__ x,
                                                               uint32_t ldx, uint32_t n,
                                                               uint32_t m_pad,
                                                               uint8_t *__restrict__ act,
                                                               wm_act_meta *__restrict__ meta) {
    __shared__ float red_f[16];
    __shared__ int red_i[16];
    const uint32_t t = blockIdx.x;
    const float *xr = x + (uint64_t)t * ldx;
    float m = 0.0f;
    for (uint32_t j = threadIdx.x; j < n; j += kRowThreads) m = wm_max_nonan(m, fabsf(xr[j]));
    const float max_abs = wm_block_max_nonan(m, red_f);
    const float inv = 127.0f / max_abs;
    int sum = 0;
    for (uint32_t j = threadIdx.x; j < n; j += kRowThreads) {
        const int q = max_abs == 0.0f ? 0 : wm_round_clamp_i8(xr[j] * inv);
        act[wm_gemm_act_offset(j, t, m_pad)] = (uint8_t)(int8_t)q;
        sum += q;
    }
    sum = wm_block_sum_i32(sum, red_i);
    if (threadIdx.x == 0) {
        meta[t].scale = max_abs == 0.0f ? 1.0f : max_abs / 127.0f;
        meta[t].asum = sum;
    }
}

// The same with a row's values read once and kept in registers: a unit is the
// 16 bytes an activation chunk holds for one weight dword (columns g + 32 q
// of a 128-column block's half, g the dword's four), four 16-byte loads and
// one 16-byte store; U units per thread.  Bound by memory: 2048 rows of 6912
// 29.4 -> 18 us (71 MB), where the kernel above reads each row twice and stores
// bytes.  For rows 16-byte aligned, of up to 4 * kRowThreads units.
template <int U>
__global__ __launch_bounds__(kRowThreads) void k_quantize_units(const float *__restrict__ x, uint32_t ldx,
                                                                uint32_t n, uint32_t m_pad,
                                                                uint8_t *__restrict__ act,
                                                                wm_act_meta *__restrict__ meta) {
    __shared__ float red_f[16];
    __shared__ int red_i[16];
    const uint32_t t = blockIdx.x, units = n / 16;
    const float *xr = x + (uint64_t)t * ldx;
    float4 v[U][4];
    float m = 0.0f;
    // unit u: chunk u / 4, dword u % 4
    const auto column = [](uint32_t u) { return (u >> 3) * 128 + ((u >> 2) & 1) * 16 + (u & 3) * 4; };
#pragma unroll
    for (int i = 0; i < U; i++) {
        const uint32_t u = threadIdx.x + i * blockDim.x;
#pragma unroll
        for (int q = 0; q < 4; q++)
            v[i][q] = u < units ? *reinterpret_cast<const float4 *>(xr + column(u) + 32 * q)
                                : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
#pragma unroll
    for (int i = 0; i < U; i++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            m = wm_max_nonan(m, fabsf(v[i][q].x));
            m = wm_max_nonan(m, fabsf(v[i][q].y));
            m = wm_max_nonan(m, fabsf(v[i][q].z));
            m = wm_max_nonan(m, fabsf(v[i][q].w));
        }
    const float max_abs = wm_block_max_nonan(m, red_f);
    const float inv = 127.0f / max_abs;
    int sum = 0;
#pragma unroll
    for (int i = 0; i < U; i++) {
        const uint32_t u = threadIdx.x + i * blockDim.x;
        if (u >= units) continue;
        uint32_t d[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float f[4] = {v[i][q].x, v[i][q].y, v[i][q].z, v[i][q].w};
            d[q] = 0;
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int c = max_abs == 0.0f ? 0 : wm_round_clamp_i8_fast(f[g] * inv);
                sum += c;
                d[q] |= (uint32_t)(uint8_t)(int8_t)c << (8 * g);
            }
        }
        *reinterpret_cast<uint4 *>(act + ((uint64_t)(u >> 2) * m_pad + t) * 64 + (u & 3) * 16) =
            make_uint4(d[0], d[1], d[2], d[3]);
    }
    sum = wm_block_sum_i32(sum, red_i);
    if (threadIdx.x == 0) {
        meta[t].scale = max_abs == 0.0f ? 1.0f : max_abs / 127.0f;
        meta[t].asum = sum;
    }
}

// ---------------------------------------------------------------------------
// RMSNorm per row (primitives.rs:227-255), one workgroup per token
// ---------------------------------------------------------------------------
// The decode norms' building blocks (wm_norm.h): the exact Σx² by the
// workgroup (seq_sum_block_owned), then y = x * rsqrt * w and the absmax
// int8 quantiser, here into the GEMM activation layout.
template <int PER, bool GU>
__global__ __launch_bounds__(kRowThreads) void k_rmsnorm_rows(wm_norm_rows a) {
    extern __shared__ __align__(16) float sq[];  // x[j]^2, seq_sum_padded(n) entries
    __shared__ wm::norm_lds<kRowThreads / 64> nl;
    const uint32_t t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, n = a.n;
    float xv[PER], wv[PER], rv[PER];
    bool nonfinite = false;
    if (GU) {
        // relu_square(gate) * up (ffn.rs:37-65)
        const float *g = a.gu + (uint64_t)t * a.ldgu;
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const uint32_t j = min(tid + (uint32_t)i * kRowThreads, n - 1);
            xv[i] = g[j];
            rv[i] = g[n + j];
            wv[i] = a.w[j];
        }
        wm::norm_prep<PER, kRowThreads>(true, n, nullptr, sq, xv, wv, rv, true);
    } else {
        float *xr = a.x + (uint64_t)t * a.ldx;
        wm::norm_load<PER, kRowThreads>(xr, a.res ? a.res + (uint64_t)t * a.ldr : nullptr, a.w, n,
                                        xv, wv, rv);
        // hidden += BitLinear output (cached_forward.rs:405-408, :496-500)
        nonfinite = wm::norm_prep<PER, kRowThreads>(a.res != nullptr, n, a.res ? xr : nullptr, sq,
                                                    xv, wv, rv);
    }
    const float rs = wm::norm_sum_rsqrt<PER, kRowThreads>(nonfinite, n, a.eps, a.err_flag, a.tag,
                                                          sq, nl);
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const uint32_t j = tid + (uint32_t)i * kRowThreads;
        xv[i] = xv[i] * rs * wv[i];
        if (j < n) {
            if (a.y_out) a.y_out[(uint64_t)t * a.ldo + j] = xv[i];
            m = wm_max_nonan(m, fabsf(xv[i]));
        }
    }
    if (!a.act) return;
    m = wm_wave_max_nonneg(m);
    if (lane == 0) nl.red_f[wid] = m;
    wm_sync_lds();
    float max_abs = nl.red_f[0];
#pragma unroll
    for (int i = 1; i < kRowThreads / 64; i++) max_abs = wm_max_nonan(max_abs, nl.red_f[i]);
    const float inv = 127.0f / max_abs;
    int sum = 0;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const uint32_t j = tid + (uint32_t)i * kRowThreads;
        if (j < n) {
            const int q = max_abs == 0.0f ? 0 : wm_round_clamp_i8_fast(xv[i] * inv);
            a.act[wm_gemm_act_offset(j, t, a.m_pad)] = (uint8_t)(int8_t)q;
            sum += q;
        }
    }
    sum = wm_wave_total_i32(sum);
    if (lane == 0) nl.red_i[wid] = sum;
    wm_sync_lds();
    if (tid == 0) {
        int tot = 0;
#pragma unroll
        for (int i = 0; i < kRowThreads / 64; i++) tot += nl.red_i[i];
        a.meta[t].scale = max_abs == 0.0f ? 1.0f : max_abs / 127.0f;
        a.meta[t].asum = tot;
    }
}

// ---------------------------------------------------------------------------
// RoPE (NEOX) + K/V append per token (cached_forward.rs:340-404)
// ---------------------------------------------------------------------------
struct qkv_rows_args {
    const float *y;
    uint32_t ldy;
    const float *cos, *sin;
    const wm_batch_tok *tok;
    uint32_t layer, n_q, n_kv, head_dim, n_rot;
    float *q_out;
};

__global__ __launch_bounds__(256) void k_qkv_rows(qkv_rows_args a) {
    extern __shared__ float sm[];  // q | k | v of this token
    __shared__ float red[16];
    const uint32_t t = blockIdx.x;
    const wm_batch_tok tk = a.tok[t];
    const uint32_t total = a.n_q + 2 * a.n_kv;
    const float *src = a.y + (uint64_t)t * a.ldy;
    for (uint32_t i = threadIdx.x; i < total; i += blockDim.x) sm[i] = src[i];
    __syncthreads();
    float *qs = sm, *ks = sm + a.n_q, *vs = ks + a.n_kv;
    const uint32_t half = a.n_rot / 2;
    const float *cs = a.cos + (uint64_t)tk.pos * half, *sn = a.sin + (uint64_t)tk.pos * half;
    const uint32_t n_pairs_q = (a.n_q / a.head_dim) * half, n_pairs_k = (a.n_kv / a.head_dim) * half;
    for (uint32_t p = threadIdx.x; p < n_pairs_q + n_pairs_k; p += blockDim.x) {
        float *base = p < n_pairs_q ? qs : ks;
        const uint32_t pp = p < n_pairs_q ? p : p - n_pairs_q;
        const uint32_t h = pp / half, j = pp % half;
        float *xh = base + h * a.head_dim;
        const float c = cs[j], s = sn[j];
        const float x0 = xh[j], x1 = xh[j + half];
        xh[j] = x0 * c - x1 * s;
        xh[j + half] = x0 * s + x1 * c;
    }
    __syncthreads();
    float *qo = a.q_out + (uint64_t)t * a.n_q;
    for (uint32_t i = threadIdx.x; i < a.n_q; i += blockDim.x) qo[i] = qs[i];
    const uint64_t row = (uint64_t)a.layer * tk.max_seq + tk.pos;
    wm_kv_quantise_store(ks, a.n_kv, tk.k + row * a.n_kv, tk.ks + row, red);
    __syncthreads();
    wm_kv_quantise_store(vs, a.n_kv, tk.v + row * a.n_kv, tk.vs + row, red);
}

// ---------------------------------------------------------------------------
// causal GQA attention of every token over its own sequence
// (cached_forward.rs:417-449, attention.rs:45-73), in three kernels
// ---------------------------------------------------------------------------
//
// Scores: one thread per (position, KV head) computes the G query heads'
// 128-term dots from one K row, each in order with k = q8 * scale, then
// * (1/sqrt(head_dim)), into scores[t][h][p].
// Softmax: per (token, head) max, exp (glibc expf), exact sequential sum,
// * (1/sum).
// V: one lane per output dimension runs Σ_p w_p * v_p[d] in position order.
struct attn_rows_args {
    const float *q;  // [t][n_heads * head_dim]
    const wm_batch_tok *tok;
    float *scores;   // [t][n_heads][score_stride]: the scores, then the weights
    float *out;      // [t][n_heads * head_dim]
    uint32_t layer, kv_dim, n_heads, score_stride, n_max;
    float scale;
    uint8_t *live;     // [t][n_heads][kAttnTiles]: the tile of kSvPos positions holds a non-zero exp
    const wm_attn_item *sc_items, *sv_items;  // work items of the scores and V kernels
};

constexpr int kScoreThreads = 256;      // positions per scores item, one per thread
constexpr uint32_t kScoreTokMax = 8;    // tokens (of one sequence) per scores item, at most

// Memory that no thread writes while the kernel runs, addressed so that the
// compiler may read it through the scalar unit wherever the address is the
// same for every lane.
typedef const float __attribute__((address_space(4))) wm_const_f32;
// Global memory, said so: a pointer read from memory is a flat one otherwise,
// and flat loads count with the scalar loads and LDS operations.
typedef const int8_t __attribute__((address_space(1))) wm_global_i8;
typedef const v4i __attribute__((address_space(1))) wm_global_v4i;
typedef const float __attribute__((address_space(1))) wm_global_f32;

// scores[t][h][p] for the nt tokens t0 .. t0+nt-1 of one sequence (item
// blockIdx.x), the G query heads of KV head `unit` and the positions p0 ..
// p0+255 below p1, one per thread: the thread dequantises its K row once
// (read_into: q8 * scale) and runs the nt*G chains Σ_i q[i] * k[i], each in
// dimension order, then * (1/sqrt(head_dim)).  Positions past a token's own
// are computed from rows other tokens of the batch have written and never
// read.
// Bound by VALU issue: each term is a separately rounded multiply and add,
// and the query values, the same for every lane, are scalar operands.  Eight
// dimensions of four rows (32 scalars) are used while the next eight are in
// flight, across the rows' ends too; read where they were used, the waits
// for them took half the time.  (As DPP broadcasts from vector registers the
// multiplies issue at 0.4 of the plain rate.)  Per BitNet-2B layer: 512
// prompt tokens from an empty cache 80 -> 32 us, 32 tokens at context 3000 69
// -> 22 (both with the placement below), 16 ragged sequences (293 tokens,
// contexts to 4000) 106 -> 94; the multiplies and adds alone take 11, 9 and
// 46 us at the rate a loop of them reaches.
template <int HD, int G>
__global__ __launch_bounds__(kScoreThreads, 2) void k_attn_scores_rows(attn_rows_args a) {
    const wm_attn_item it = a.sc_items[blockIdx.x];
    const uint32_t p = it.p0 + threadIdx.x;
    if (it.nt == 0 || (p & ~63u) >= it.p1) return;  // (p0 is a multiple of 64: whole waves)
    const uint32_t kvh = it.unit, rows = it.nt * G;
    const wm_batch_tok tk = a.tok[it.t0];  // every token of the item: the same cache
    const uint64_t lay = (uint64_t)a.layer * tk.max_seq;
    // row r: head r % G of token r / G; four rows at a time (a row past the
    // last: the last again, not stored)
    const wm_const_f32 *q0 = (const wm_const_f32 *)a.q + ((uint64_t)it.t0 * a.n_heads + kvh * G) * HD;
    const auto row_off = [&](uint32_t r) { return (uint64_t)(r / G) * a.n_heads + r % G; };
    const uint32_t r_last = (rows - 1) & ~3u;
    struct q_block {
        float v[4][8];
    };
    const auto q_load = [&](q_block &q, uint32_t r0, int d) {
        const wm_const_f32 *qr[4];
        if constexpr (G % 4 == 0) {  // heads of one token: consecutive rows
            qr[0] = q0 + row_off(r0) * HD + d;
            // (opaque, so that two blocks' loads are not merged: the scalar
            // registers hold two blocks, not four)
            asm volatile("" : "+s"(qr[0]));
#pragma unroll
            for (uint32_t i = 1; i < 4; i++) qr[i] = qr[0] + i * HD;
        } else {
#pragma unroll
            for (uint32_t i = 0; i < 4; i++) {
                qr[i] = q0 + row_off(min(r0 + i, rows - 1)) * HD + d;
                asm volatile("" : "+s"(qr[i]));
            }
        }
#pragma unroll
        for (uint32_t i = 0; i < 4; i++)
#pragma unroll
            for (int e = 0; e < 8; e++) q.v[i][e] = qr[i][e];
    };
    q_block qa, qb;
    q_load(qa, 0, 0);
    float kd[HD];
    {
        const uint32_t pc = min(p, it.p1 - 1);  // (a thread past the end computes the last position, not stored)
        const wm_global_v4i *kp = (const wm_global_v4i *)(tk.k + (lay + pc) * a.kv_dim + kvh * HD);
        const float kscale = ((const wm_global_f32 *)tk.ks)[lay + pc];
        v4i raw[HD / 16];
#pragma unroll
        for (int b = 0; b < HD / 16; b++) raw[b] = kp[b];
#pragma unroll
        for (int i = 0; i < HD; i++) {
            const v4i c = raw[i / 16];
            const int e = i % 16;
            const uint32_t wd = e < 4 ? (uint32_t)c.x : e < 8 ? (uint32_t)c.y : e < 12 ? (uint32_t)c.z : (uint32_t)c.w;
            kd[i] = (float)(int8_t)(wd >> (8 * (e & 3))) * kscale;  // read_into
        }
    }
    float *dst = a.scores + ((uint64_t)it.t0 * a.n_heads + kvh * G) * a.score_stride + p;
#pragma unroll 1
    for (uint32_t r0 = 0; r0 < rows; r0 += 4) {
        float s[4];
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) s[i] = 0.0f;
        const auto add8 = [&](const q_block &q, int d) {
#pragma unroll
            for (int e = 0; e < 8; e++)
#pragma unroll
                for (uint32_t i = 0; i < 4; i++) s[i] = s[i] + q.v[i][e] * kd[d + e];
            __builtin_amdgcn_sched_barrier(0);
        };
        // Scalar loads return in any order, so a wait for one is a wait for
        // all: the block about to be used is waited for (it had the block
        // before it to arrive) before the next one's loads go out.
        const auto wait_q = [&]() {
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0) alone
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int d = 0; d < HD; d += 16) {
            wait_q();
            q_load(qb, r0, d + 8);
            __builtin_amdgcn_sched_barrier(0);  // the loads go out before these terms
            add8(qa, d);
            wait_q();
            if (d + 16 < HD) q_load(qa, r0, d + 16);
            else q_load(qa, min(r0 + 4, r_last), 0);  // the next rows'
            __builtin_amdgcn_sched_barrier(0);
            add8(qb, d + 8);
        }
        // (the chains end here, not inside the branch)
        asm volatile("" : "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3]));
        if (p < it.p1)
#pragma unroll
            for (uint32_t i = 0; i < 4; i++)
                if (r0 + i < rows) dst[row_off(r0 + i) * a.score_stride] = s[i] * a.scale;
    }
}

constexpr uint32_t kSvPos = WM_ATTN_TILE;  // positions per tile of the V pass
constexpr uint32_t kAttnTiles = 64;  // tiles per row (contexts <= 4096)
constexpr uint32_t kSvDimRow = 20;   // dwords of a dimension's 64 codes of a tile in LDS (spread banks)

// Softmax of the scores rows in place (attention.rs:45-73): max, exp (glibc
// expf), the exact sequential sum of the exps, and each weight exp * (1/sum)
// (the exp itself when the sum is not positive: the reference leaves the row
// unnormalised); zeros from the row's end to the end of its tile of kSvPos
// positions.  Tiles whose exps are all exactly zero are flagged dead: their
// weights are zero, and a zero term leaves each of the V pass's sums
// unchanged (those sums start at +0 and can never be -0), so it skips them.
// A row whose maximum is not finite becomes all zero (its output is then 0).
//
// A row's values stay in the registers of its WPR waves (F4 float4 a lane: n
// <= 256 WPR F4).  The sum is the plain chain of adds: 1024 positions of every
// row at a time go through LDS, and wave 0 adds the workgroup's rows side by
// side, a quarter of its lanes per row, four terms per LDS read, while the
// next 1024 positions' exps are formed.  The chain costs ~2.4 ns a term and one
// VALU slot for all the rows; the integer sum per 512-term step it replaces
// restarts at every binade change and halfway case, several hundred cycles
// each.  Per BitNet-2B layer (rows x mean context): 10220 x 256 25.8 -> 12.5
// us, 640 x 3000 25.6 -> 18.4, 5860 x 2000 55 -> 50.
// (exp of a score minus its row's maximum, so of x <= 0 or a NaN: expf_glibc
// without its branches.  Below -0x1.9fe368p6 it is +0.)
__device__ __forceinline__ float exp_nonpos(float x, const uint64_t *tab) {
    const float y = wm::expf_glibc_core(x < -104.0f ? -104.0f : x, tab);
    return x < -0x1.9fe368p6f ? 0.0f : y;
}
constexpr uint32_t kSmRows = 4;      // rows per workgroup
constexpr uint32_t kSmChunk = 1024;  // positions of each row in LDS at a time
template <uint32_t WPR, uint32_t F4>
__global__ __launch_bounds__(kSmRows * WPR * 64) void k_attn_softmax_rows(attn_rows_args a, uint32_t n_rows) {
    constexpr uint32_t kSlots = kSmChunk / 256;  // float4 slots of a chunk
    constexpr uint32_t kMine = kSlots / WPR;     // a wave's slots of a chunk
    constexpr uint32_t kChunks = (F4 + kMine - 1) / kMine;
    constexpr uint32_t kBufs = kChunks > 1 ? 2 : 1;
    static_assert(kSlots % WPR == 0, "a chunk's slots over the row's waves");
    __shared__ __align__(16) float buf[kBufs][kSmRows][kSmChunk + 4];  // (rows on different banks)
    __shared__ uint64_t exp_tab[32];
    __shared__ float row_inv[kSmRows], red[kSmRows * WPR];
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wid = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t r = wid / WPR, part = wid % WPR;  // row of the workgroup, the wave's part of it
    const uint32_t row0 = blockIdx.x * kSmRows, row = min(row0 + r, n_rows - 1);
    const bool mine = row0 + r < n_rows;
    const uint32_t n = a.tok[row / a.n_heads].pos + 1;
    float *w = a.scores + (uint64_t)row * a.score_stride;
    // Slot k: positions 256 k + 4 lane .. + 3, of wave k % WPR.  (Rows are
    // padded to whole tiles, so a float4 that holds a position below n lies
    // inside the row; indices are clamped to the last such one.)
    const uint32_t n4 = (n + 3) / 4;
    float4 x[F4];
#pragma unroll
    for (uint32_t i = 0; i < F4; i++) {
        const uint32_t k = i * WPR + part;
        if (256 * k < n) x[i] = reinterpret_cast<const float4 *>(w)[min(64 * k + lane, n4 - 1)];
    }
    uint32_t n_max = 0;  // the workgroup's longest row (its rows are of one token or of a few)
#pragma unroll
    for (uint32_t i = 0; i < kSmRows; i++)
        n_max = max(n_max, a.tok[min(row0 + i, n_rows - 1) / a.n_heads].pos + 1);
    if (tid < 32) exp_tab[tid] = wm::kExp2Tab[tid];
    float mx = -INFINITY;
#pragma unroll
    for (uint32_t i = 0; i < F4; i++) {
        const uint32_t k = i * WPR + part;
        if (256 * k < n) {
            const uint32_t p = 256 * k + 4 * lane;
            mx = wm_max_nonan(mx, p < n ? x[i].x : -INFINITY);
            mx = wm_max_nonan(mx, p + 1 < n ? x[i].y : -INFINITY);
            mx = wm_max_nonan(mx, p + 2 < n ? x[i].z : -INFINITY);
            mx = wm_max_nonan(mx, p + 3 < n ? x[i].w : -INFINITY);
        }
    }
    mx = wm_wave_max_nonan(mx);
    if (WPR > 1 && lane == 0) red[wid] = mx;
    __syncthreads();
    if (WPR > 1)
#pragma unroll
        for (uint32_t i = 0; i < WPR; i++) mx = wm_max_nonan(mx, red[r * WPR + i]);
    const bool zero = !isfinite(mx);  // every weight becomes 0 (or the row held a NaN)
    float s = 0.0f;                   // wave 0: the sum of row lane / 16
    // this wave's part of chunk c: exps in place and into LDS (zeros past a
    // shorter row's end change nothing)
    const auto exps = [&](uint32_t c) {
#pragma unroll
        for (uint32_t u = 0; u < kMine; u++) {
            const uint32_t i = c * kMine + u, k = i * WPR + part;
            float4 e = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (i < F4 && 256 * k < n) {
                const uint32_t p = 256 * k + 4 * lane;
                float4 &v = x[i < F4 ? i : 0];
                if (!zero) {
                    e.x = p < n ? exp_nonpos(v.x - mx, exp_tab) : 0.0f;
                    e.y = p + 1 < n ? exp_nonpos(v.y - mx, exp_tab) : 0.0f;
                    e.z = p + 2 < n ? exp_nonpos(v.z - mx, exp_tab) : 0.0f;
                    e.w = p + 3 < n ? exp_nonpos(v.w - mx, exp_tab) : 0.0f;
                }
                v = e;
                // lanes 16 j .. 16 j + 15 hold tile 4 k + j
                const uint64_t nz = __ballot(e.x != 0.0f || e.y != 0.0f || e.z != 0.0f || e.w != 0.0f);
                if (mine && lane < 4 && (4 * k + lane) * kSvPos < n)
                    a.live[(uint64_t)row * kAttnTiles + 4 * k + lane] = (nz >> (16 * lane) & 0xFFFFu) != 0 ? 1 : 0;
            }
            *reinterpret_cast<float4 *>(&buf[c % kBufs][r][256 * (k % kSlots) + 4 * lane]) = e;
        }
    };
    const auto chain = [&](uint32_t c) {
        const float *src = buf[c % kBufs][lane / 16];
        const uint32_t m = min(kSmChunk, n_max - c * kSmChunk);
        // 32 terms per step, each half's reads ahead of the other's adds
        float4 f[2][4];
        const auto read16 = [&](float4 (&g)[4], uint32_t q) {
#pragma unroll
            for (uint32_t i = 0; i < 4; i++) g[i] = *reinterpret_cast<const float4 *>(src + q + 4 * i);
            __builtin_amdgcn_sched_barrier(0);
        };
        const auto add16 = [&](const float4 (&g)[4]) {
#pragma unroll
            for (uint32_t i = 0; i < 4; i++) {
                s = s + g[i].x;
                s = s + g[i].y;
                s = s + g[i].z;
                s = s + g[i].w;
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        read16(f[0], 0);
        __builtin_amdgcn_s_setprio(3);  // (the chain's wave first on its SIMD: the others wait for it)
#pragma unroll 1
        for (uint32_t q = 0; q < m; q += 32) {
            // (what a step adds past m is zeros; past the chunk nothing is read)
            read16(f[1], q + 16);
            add16(f[0]);
            read16(f[0], q + 32 < kSmChunk ? q + 32 : 0u);
            add16(f[1]);
        }
        __builtin_amdgcn_s_setprio(0);
    };
    exps(0);
#pragma unroll
    for (uint32_t c = 0; c < kChunks; c++) {
        if (c * kSmChunk >= n_max) break;
        __syncthreads();  // chunk c is in LDS; chunk c - 1 is summed
        if (c + 1 < kChunks && (c + 1) * kSmChunk < n_max) exps(c + 1);
        if (wid == 0) chain(c);
    }
    if (wid == 0 && lane % 16 == 0) row_inv[lane / 16] = s > 0.0f ? 1.0f / s : 1.0f;
    __syncthreads();
    if (!mine) return;
    const float inv = row_inv[r];
    const uint32_t end = (n + kSvPos - 1) / kSvPos * kSvPos;
#pragma unroll
    for (uint32_t i = 0; i < F4; i++) {
        const uint32_t p = 256 * (i * WPR + part) + 4 * lane;
        if (p < end)
            *reinterpret_cast<float4 *>(w + p) = make_float4(x[i].x * inv, x[i].y * inv, x[i].z * inv, x[i].w * inv);
    }
}

// One wave's LDS operations complete in order; the compiler keeps that order
// across this point.
__device__ __forceinline__ void wave_lds_order() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
}

// One wave's part of k_attn_sv_rows: out[h][d] for its 64 dimensions (lane =
// one of them) of the heads of one token, C at a time: heads 0 .. C-1 over the
// tiles of ms[0], the next C over those of ms[1], and so on for all N masks
// (w, out: head 0's weights and outputs).  The next tile's codes, weights and
// scales are in flight behind the one in use, across the heads' ends too; the
// weights and V scales, the same for every lane, go through LDS (wts, my: the
// wave's own) as broadcasts, four positions per read, read ahead of use.
template <int HD, int C, int N>
__device__ __forceinline__ void sv_heads(const attn_rows_args &a, const wm_global_i8 *vg, const wm_global_f32 *vs,
                                         const wm_global_f32 *w, float *out, float (*wts)[kSvPos], uint32_t *my,
                                         uint64_t (&ms)[N]) {
    const uint32_t lane = threadIdx.x & 63;
    float acc[C];
#pragma unroll
    for (int c = 0; c < C; c++) acc[c] = 0.0f;

    // A tile as loaded.  Codes: lane 16 s + g takes dimensions 4 g .. 4 g+3 (a
    // dword) of positions 16 i + 4 s + j, dword 4 i + j.  The
    // heads' weights and the V scale of position `lane`.
    // (Positions from n to the tile's end have zero weights.  Their codes and
    // scales are whatever the cache holds there, always finite: it is
    // allocated a tile longer and its scales start as zeros.)
    struct tile_regs {
        uint32_t v[16];
        float x[C + 1];
    };
    uint32_t v_off[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) v_off[j] = (4 * (lane >> 4) + j) * a.kv_dim + 4 * (lane & 15);
    const auto fetch = [&](tile_regs &q, uint32_t h, uint32_t p) {
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
            const wm_global_i8 *vp = vg + (uint64_t)(p + 16 * i) * a.kv_dim;
            asm volatile("" : "+s"(vp));
#pragma unroll
            for (uint32_t j = 0; j < 4; j++) {
                // (opaque: its widening stays at the load, which then takes a
                // scalar base and this 32-bit offset)
                asm volatile("" : "+v"(v_off[j]));
                q.v[4 * i + j] = *(const uint32_t __attribute__((address_space(1))) *)(vp + v_off[j]);
            }
        }
#pragma unroll
        for (uint32_t c = 0; c < (uint32_t)C; c++) q.x[c] = w[(uint64_t)(h + c) * a.score_stride + p + lane];
        q.x[C] = vs[p + lane];
        __builtin_amdgcn_sched_barrier(0);
    };
    // Each dimension's 64 codes to its lane, through LDS: four positions'
    // bytes of a dimension per dword (4 x 4 byte transposes), lane d reads
    // slots s of dwords i: positions 16 i + 4 s ..  (A dimension's slots are
    // XORed with its bits 5:4, so that eight lanes' accesses share no bank.)
    const auto turn = [&](const tile_regs &q, uint32_t (&o)[16]) {
#pragma unroll
        for (int c = 0; c <= C; c++) wts[c][lane] = q.x[c];
        uint32_t td[4][4];  // [dimension][i]
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
            const uint32_t x0 = q.v[4 * i], x1 = q.v[4 * i + 1], x2 = q.v[4 * i + 2], x3 = q.v[4 * i + 3];
            const uint32_t a01 = __builtin_amdgcn_perm(x1, x0, 0x05010400u), b01 = __builtin_amdgcn_perm(x1, x0, 0x07030602u);
            const uint32_t a23 = __builtin_amdgcn_perm(x3, x2, 0x05010400u), b23 = __builtin_amdgcn_perm(x3, x2, 0x07030602u);
            td[0][i] = __builtin_amdgcn_perm(a23, a01, 0x05040100u);
            td[1][i] = __builtin_amdgcn_perm(a23, a01, 0x07060302u);
            td[2][i] = __builtin_amdgcn_perm(b23, b01, 0x05040100u);
            td[3][i] = __builtin_amdgcn_perm(b23, b01, 0x07060302u);
        }
#pragma unroll
        for (uint32_t d = 0; d < 4; d++)
            *reinterpret_cast<uint4 *>(my + (4 * (lane & 15) + d) * kSvDimRow + 4 * ((lane >> 4) ^ ((lane >> 2) & 3))) =
                make_uint4(td[d][0], td[d][1], td[d][2], td[d][3]);
        wave_lds_order();
#pragma unroll
        for (uint32_t s = 0; s < 4; s++) {
            const uint4 r = *reinterpret_cast<const uint4 *>(my + lane * kSvDimRow + 4 * (s ^ (lane >> 4)));
            o[s] = r.x;  // dword 4 i + s: positions 16 i + 4 s .. + 3
            o[4 + s] = r.y;
            o[8 + s] = r.z;
            o[12 + s] = r.w;
        }
        wave_lds_order();
    };
    constexpr uint32_t kL = C == 4 ? 4 : 8;  // positions read ahead
    struct block {
        float4 w[C][kL / 4], s[kL / 4];
    };
    const auto read = [&](block &q, uint32_t e) {
#pragma unroll
        for (uint32_t i = 0; i < kL / 4; i++) {
            q.s[i] = *reinterpret_cast<const float4 *>(&wts[C][e + 4 * i]);
#pragma unroll
            for (int c = 0; c < C; c++) q.w[c][i] = *reinterpret_cast<const float4 *>(&wts[c][e + 4 * i]);
        }
        __builtin_amdgcn_sched_barrier(0);  // the reads go out before the terms that follow
    };
    const auto pick = [](const float4 &x, uint32_t e) { return e == 0 ? x.x : e == 1 ? x.y : e == 2 ? x.z : x.w; };
    const auto add = [&](const block &q, const uint32_t (&v)[16], uint32_t e0) {
#pragma unroll
        for (uint32_t e = 0; e < kL; e++) {
            const float f = (float)(int8_t)(v[(e0 + e) / 4] >> (8 * (e % 4))) * pick(q.s[e / 4], e % 4);  // read_into
#pragma unroll
            for (int c = 0; c < C; c++) acc[c] = acc[c] + pick(q.w[c][e / 4], e % 4) * f;
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    const auto store = [&](uint32_t h) {
#pragma unroll
        for (uint32_t c = 0; c < (uint32_t)C; c++) {
            out[(h + c) * HD + lane] = acc[c];
            acc[c] = 0.0f;
        }
    };
    const auto remain = [&]() {
        uint64_t m = ms[0];
#pragma unroll
        for (int i = 1; i < N; i++) m |= ms[i];
        return m != 0;
    };
    // the heads of the next tile: those without one are left out
    uint32_t h_next = 0;
    const auto next_head = [&]() {  // (a mask is not empty)
#pragma unroll
        for (int i = 1; i < N; i++)
            if (ms[0] == 0) {
#pragma unroll
                for (int k = 1; k < N; k++) ms[k - 1] = ms[k];
                ms[N - 1] = 0;
                h_next += C;
            }
    };
    const auto next_tile = [&]() {
        const uint32_t r = (uint32_t)__builtin_ctzll(ms[0]) * kSvPos;
        ms[0] &= ms[0] - 1;
        return r;
    };
#pragma unroll
    for (uint32_t i = 0; N > 1 && i < (uint32_t)N; i++)
        if (ms[i] == 0) store(i * C);
    if (remain()) {
        tile_regs cur;
        uint32_t v[16];
        block qa, qb;
        next_head();
        uint32_t h = h_next;  // the heads of the tile in use
        fetch(cur, h, next_tile());
        for (bool more = true; more;) {
            turn(cur, v);
            read(qa, 0);
            more = remain();
            if (more) {
                next_head();
                fetch(cur, h_next, next_tile());
            }
#pragma unroll
            for (uint32_t e = 0; e < kSvPos; e += 2 * kL) {
                read(qb, e + kL);
                add(qa, v, e);
                if (e + 2 * kL < kSvPos) read(qa, e + 2 * kL);
                add(qb, v, e + kL);
            }
            wave_lds_order();  // the tile's weights are read
            if (N > 1 && (!more || h_next != h)) {
                store(h);
                h = h_next;
            }
        }
    }
    if (N == 1) store(0);
}

// out[t][h][d] = Σ_p w_h[p] * v_p[d] in position order (cached_forward.rs:
// 417-449; v_p[d] = q8 * scale, read_into), w the softmax's weights.  A wave
// runs C query heads of one KV head for one token ("row set"), lane = one of
// 64 dimensions, over the row set's live tiles: together, the heads sharing
// each dequantised value (a tile dead for some of them adds zeros to those),
// or, where their live tiles are mostly different ones, one head after the
// other, each over its own.
// Bound by VALU issue, 2 C + 2 instructions per position, and by the longest
// rows: a wave issues one instruction in ~4 cycles at best, so they go first
// (item order, s_setprio).  Other ways to a weight: as a scalar operand the
// load takes ~750 cycles, more than 32 scalars in flight cover (173-181 us at
// the ragged shape below); as a DPP broadcast the multiply issues at 0.4 of
// its rate; a readlane takes three slots; products from a 4 x 4 x 1 MFMA
// (exact, four rows at once) took 178.  The kernel it replaces ran one head per
// workgroup, a byte read from LDS per position and lane.  Per BitNet-2B layer:
// 512 prompt tokens 70 -> 36 us, 32 tokens at context 3000 74 -> 67, 16 ragged
// sequences (293 tokens) 275 -> 159.  Where the softmaxes are sparse (16 ragged
// sequences, 257 tokens, N(0,1) K and V: most rows one live tile, some all) a
// wave over its heads' tiles together took 99 us, the kernel before it 90, one
// head after the other where that is shorter 87; the choice costs dense rows
// under 1 % (36, 68 and 157 us at the shapes above).
template <int HD, int C>
__global__ __launch_bounds__(256) void k_attn_sv_rows(attn_rows_args a, uint32_t group) {
    constexpr uint32_t NH = HD / 64;  // waves per row set
    __shared__ __align__(16) uint32_t lds[4][64 * kSvDimRow];
    __shared__ __align__(16) float wts[4][C + 1][kSvPos];  // the tile's weights, V scales
    const wm_attn_item it = a.sv_items[blockIdx.x];
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wid = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (wid / NH >= it.nt) return;
    const uint32_t rs = it.p0 + wid / NH, per = group / C;  // row set, row sets per token
    const uint32_t t = it.t0 + rs / per, h0 = it.unit * group + rs % per * C;
    const wm_batch_tok tk = a.tok[t];
    const uint32_t n = tk.pos + 1;
    const uint64_t row = (uint64_t)t * a.n_heads + h0;
    // the tiles where each head, and where any of them, has a non-zero weight
    uint32_t lv[C];
#pragma unroll
    for (uint32_t c = 0; c < (uint32_t)C; c++)
        lv[c] = a.live[(row + c) * kAttnTiles + min(lane, (n - 1) / kSvPos)];
    const uint32_t in = lane * kSvPos < n ? 1u : 0u;
    uint64_t own[C], any[1] = {0};
    uint32_t tiles = 0;
#pragma unroll
    for (uint32_t c = 0; c < (uint32_t)C; c++) {
        own[c] = __ballot((lv[c] & in) != 0);
        any[0] |= own[c];
        tiles += (uint32_t)__builtin_popcountll(own[c]);
    }
    const uint32_t shared = (uint32_t)__builtin_popcountll(any[0]);
    const uint64_t lay = (uint64_t)a.layer * tk.max_seq;
    const uint32_t d0 = (wid % NH) * 64;
    const wm_global_i8 *vg = (const wm_global_i8 *)tk.v + lay * a.kv_dim + it.unit * HD + d0;
    const wm_global_f32 *vs = (const wm_global_f32 *)tk.vs + lay;
    const wm_global_f32 *w = (const wm_global_f32 *)a.scores + row * a.score_stride;
    float *out = a.out + row * HD + d0;
    // The longest rows end last: their waves go first on their SIMDs.
    const uint32_t q = n * 4 / a.n_max;
    if (q >= 3) __builtin_amdgcn_s_setprio(3);
    else if (q == 2) __builtin_amdgcn_s_setprio(2);
    else if (q == 1) __builtin_amdgcn_s_setprio(1);
    // By the instructions of a tile: about C + 2 units with C heads at once, 3
    // with one (~100 for the tile's codes and 64 (2 C + 2) + 17 (C + 1)).
    if (C > 1 && tiles * 3 < shared * (C + 2)) sv_heads<HD, 1, C>(a, vg, vs, w, out, wts[wid], lds[wid], own);
    else sv_heads<HD, C, 1>(a, vg, vs, w, out, wts[wid], lds[wid], any);
}

}  // namespace

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------

namespace {
constexpr uint32_t kGemmCus = 256;
constexpr uint32_t kAttnSimds = 4 * kGemmCus;
}  // namespace

wm_gemm_plan wm_gemm_make_plan(uint32_t groups, uint32_t n_chunks, uint32_t m) {
    (void)n_chunks;
    wm_gemm_plan p;
    p.tiles = (m + WM_GEMM_TILE_TOKENS - 1) / WM_GEMM_TILE_TOKENS;
    // Up to two 64 x 64 output tiles per CU: the waves split K
    // (k_i2s_gemm_kw, 3 chunks in flight per wave; two workgroups fit a
    // CU's LDS).  More: the waves split the tokens of two groups per
    // workgroup (k_i2s_gemm, double-buffered).  These were the faster
    // choices in a sweep of both kernels, NG and ring depth over the
    // BitNet-2B shapes at M = 257.
    if (groups * p.tiles <= 2 * kGemmCus) {
        p.kw = true;
        p.ng = 1;
        p.st = 3;
    } else {  // more than 512 tiles: at least 256 workgroups of two groups
        p.ng = 2;
        p.st = 2;
    }
    p.gx = (groups + p.ng - 1) / p.ng;
    return p;
}

bool wm_launch_i2s_gemm(const wm_gemm_desc *d, int n_desc, uint32_t n_chunks, const uint8_t *act,
                        uint32_t m, uint32_t m_pad, const wm_act_meta *meta, float *y,
                        uint32_t ldy, hipStream_t s) {
    gemm_args a{};
    uint32_t groups = 0;
    for (int i = 0; i < n_desc; i++) {
        a.d[i] = d[i];
        groups += d[i].n_groups;
        a.group_end[i] = groups;
    }
    a.n_desc = n_desc;
    a.n_groups = groups;
    a.n_chunks = n_chunks;
    a.act = act;
    a.m = m;
    a.m_pad = m_pad;
    a.meta = meta;
    a.y = y;
    a.ldy = ldy;
    const wm_gemm_plan p = wm_gemm_make_plan(groups, n_chunks, m);
    const dim3 grid(p.gx, p.tiles);
#define WM_GEMM_CASE(KW, NG, ST)                                                                 \
    if (p.kw == KW && p.ng == NG && p.st == ST) {                                                \
        if (KW)                                                                                  \
            hipLaunchKernelGGL((k_i2s_gemm_kw<NG, ST>), grid, dim3(256), (gemm_kw_lds_bytes<NG, ST>()), s, a); \
        else                                                                                     \
            hipLaunchKernelGGL((k_i2s_gemm<NG, ST>), grid, dim3(256), (gemm_lds_bytes<NG, ST>()), s, a); \
        return true;                                                                             \
    }
    WM_GEMM_CASE(true, 1, 3)
    WM_GEMM_CASE(false, 2, 2)
#undef WM_GEMM_CASE
    return false;  // a plan with no instantiation: nothing launched
}

void wm_launch_quantize_rows(const float *x, uint32_t ldx, uint32_t n, uint32_t m, uint32_t m_pad,
                             uint8_t *act, wm_act_meta *meta, hipStream_t s) {
    const uint32_t units = n / 16;
    if (n % 128 == 0 && ((uintptr_t)x & 15) == 0 && ldx % 4 == 0 && units <= 4 * kRowThreads) {
        const uint32_t threads = std::min<uint32_t>(kRowThreads, (units + 63) / 64 * 64);
        if (units <= threads)
            hipLaunchKernelGGL(k_quantize_units<1>, dim3(m), dim3(threads), 0, s, x, ldx, n, m_pad, act, meta);
        else if (units <= 2 * threads)
            hipLaunchKernelGGL(k_quantize_units<2>, dim3(m), dim3(threads), 0, s, x, ldx, n, m_pad, act, meta);
        else
            hipLaunchKernelGGL(k_quantize_units<4>, dim3(m), dim3(threads), 0, s, x, ldx, n, m_pad, act, meta);
        return;
    }
    hipLaunchKernelGGL(k_quantize_rows, dim3(m), dim3(kRowThreads), 0, s, x, ldx, n, m_pad, act,
                       meta);
}

bool wm_launch_rmsnorm_rows(const wm_norm_rows &a, uint32_t m, hipStream_t s) {
    const size_t lds = (size_t)wm::seq_sum_padded(a.n) * sizeof(float);
    const int per = (int)((a.n + kRowThreads - 1) / kRowThreads);
    const bool gu = a.gu != nullptr;
#define WM_ROWS_CASE(P)                                                                          \
    case P:                                                                                      \
        if (gu) hipLaunchKernelGGL((k_rmsnorm_rows<P, true>), dim3(m), dim3(kRowThreads), lds, s, a); \
        else hipLaunchKernelGGL((k_rmsnorm_rows<P, false>), dim3(m), dim3(kRowThreads), lds, s, a);   \
        return true;
    switch (per) {
        WM_ROWS_CASE(1) WM_ROWS_CASE(2) WM_ROWS_CASE(3) WM_ROWS_CASE(4)
        WM_ROWS_CASE(5) WM_ROWS_CASE(6) WM_ROWS_CASE(7) WM_ROWS_CASE(8)
        WM_ROWS_CASE(9) WM_ROWS_CASE(10) WM_ROWS_CASE(11) WM_ROWS_CASE(12)
        WM_ROWS_CASE(13) WM_ROWS_CASE(14) WM_ROWS_CASE(15) WM_ROWS_CASE(16)
        default: break;
    }
#undef WM_ROWS_CASE
    return false;  // n above 8192: no instantiation
}

void wm_launch_qkv_rows(const float *y, uint32_t ldy, const float *rope_cos, const float *rope_sin,
                        const wm_batch_tok *tok, uint32_t m, uint32_t layer, uint32_t n_q,
                        uint32_t n_kv, uint32_t head_dim, uint32_t n_rot, float *q_out,
                        hipStream_t s) {
    qkv_rows_args a{y, ldy, rope_cos, rope_sin, tok, layer, n_q, n_kv, head_dim, n_rot, q_out};
    const size_t lds = (size_t)(n_q + 2 * n_kv) * sizeof(float);
    hipLaunchKernelGGL(k_qkv_rows, dim3(m), dim3(256), lds, s, a);
}

bool wm_attn_rows_supported(uint32_t head_dim, uint32_t group) {
    return (head_dim == 64 || head_dim == 128) &&
           (group == 1 || group == 2 || group == 4 || group == 8);
}

// scores [m][n_heads][stride] (whole tiles) | live tiles [m][n_heads][kAttnTiles]
static uint32_t attn_stride(uint32_t n_max) { return (n_max + kSvPos - 1) / kSvPos * kSvPos; }
static size_t attn_scores_part(uint32_t m, uint32_t n_heads, uint32_t n_max) {
    return ((size_t)m * n_heads * attn_stride(n_max) * sizeof(float) + 255) & ~(size_t)255;
}
static size_t attn_live_part(uint32_t m, uint32_t n_heads) {
    return ((size_t)m * n_heads * kAttnTiles + 255) & ~(size_t)255;
}
size_t wm_attn_rows_scores_bytes(uint32_t m, uint32_t n_heads, uint32_t n_max, uint32_t n_items) {
    return attn_scores_part(m, n_heads, n_max) + attn_live_part(m, n_heads) + (size_t)n_items * sizeof(wm_attn_item);
}
wm_attn_item *wm_attn_rows_items(float *scores, uint32_t m, uint32_t n_heads, uint32_t n_max) {
    return reinterpret_cast<wm_attn_item *>(reinterpret_cast<uint8_t *>(scores) +
                                            attn_scores_part(m, n_heads, n_max) +
                                            attn_live_part(m, n_heads));
}

// Workgroup i runs on XCD i % 8.  The items of one (sequence, unit) read the
// same K or V rows, so they share an XCD's L2 while that leaves the XCDs
// evenly loaded: a group of items is cut into pieces of at most 1/32 of the
// work, and each piece goes to the least-loaded XCD, largest first (a single
// sequence has one group per KV head: uncut, its five groups left three XCDs
// idle).  An XCD's items run in order of their work, the longest first; the
// shorter lists are padded with empty items.
struct attn_piece {
    uint64_t work;
    uint32_t first, n;  // items [first, first + n)
};
static void attn_place(const std::vector<wm_attn_item> &items, const std::vector<uint64_t> &work,
                       const std::vector<uint32_t> &group, std::vector<wm_attn_item> &out) {
    constexpr uint32_t kXcds = 8, kPieces = 32;
    uint64_t total = 0;
    for (uint64_t w : work) total += w;
    std::vector<attn_piece> pieces;
    for (uint32_t i = 0; i < items.size(); i++) {
        if (i == 0 || group[i] != group[i - 1] || (pieces.back().work + work[i]) * kPieces > total)
            pieces.push_back({0, i, 0});
        pieces.back().work += work[i];
        pieces.back().n++;
    }
    std::stable_sort(pieces.begin(), pieces.end(),
                     [](const attn_piece &x, const attn_piece &y) { return x.work > y.work; });
    std::vector<uint32_t> lists[kXcds];
    uint64_t load[kXcds] = {};
    for (const attn_piece &p : pieces) {
        uint32_t x = 0;
        for (uint32_t k = 1; k < kXcds; k++)
            if (load[k] < load[x]) x = k;
        load[x] += p.work;
        for (uint32_t i = 0; i < p.n; i++) lists[x].push_back(p.first + i);
    }
    size_t len = 0;
    for (auto &l : lists) {
        std::stable_sort(l.begin(), l.end(), [&](uint32_t x, uint32_t y) { return work[x] > work[y]; });
        len = std::max(len, l.size());
    }
    out.assign(len * kXcds, wm_attn_item{0, 0, 0, 0, 0, 0});
    for (uint32_t x = 0; x < kXcds; x++)
        for (size_t k = 0; k < lists[x].size(); k++) out[k * kXcds + x] = items[lists[x][k]];
}

uint32_t wm_attn_rows_plan(const wm_batch_tok *tok, uint32_t m, uint32_t n_kv_heads, uint32_t group,
                           uint32_t head_dim, std::vector<wm_attn_item> &sc, std::vector<wm_attn_item> &sv) {
    // the sequences: tokens of one cache at consecutive positions
    std::vector<std::pair<uint32_t, uint32_t>> seqs;
    for (uint32_t t = 0; t < m;) {
        uint32_t e = t + 1;
        while (e < m && tok[e].k == tok[t].k && tok[e].pos == tok[e - 1].pos + 1) e++;
        seqs.emplace_back(t, e);
        t = e;
    }
    // Tokens per scores item: as many as leave three waves per SIMD (a K row
    // is dequantised once per item, its share small from four tokens on).
    uint32_t nt_max = kScoreTokMax;
    for (; nt_max > 1; nt_max /= 2) {
        uint64_t waves = 0;
        for (auto &q : seqs)
            for (uint32_t b = q.first; b < q.second; b += nt_max)
                waves += (uint64_t)n_kv_heads * (tok[std::min(b + nt_max, q.second) - 1].pos / 64 + 1);
        if (waves >= 3 * kAttnSimds) break;
    }
    std::vector<wm_attn_item> items;
    std::vector<uint64_t> work;
    std::vector<uint32_t> gids;
    uint32_t gid = 0;
    for (auto &q : seqs)
        for (uint32_t u = 0; u < n_kv_heads; u++, gid++)
            for (uint32_t b = q.first; b < q.second; b += nt_max) {
                const uint32_t nt = std::min(nt_max, q.second - b), p1 = tok[b + nt - 1].pos + 1;
                for (uint32_t p0 = 0; p0 < p1; p0 += kScoreThreads) {
                    items.push_back({b, nt, p0, p1, u, 0});
                    work.push_back((uint64_t)nt * std::min<uint32_t>(kScoreThreads, p1 - p0));
                    gids.push_back(gid);
                }
            }
    attn_place(items, work, gids, sc);
    items.clear();
    work.clear();
    gids.clear();
    // V kernel: the most query heads per wave that leave four waves per SIMD,
    // else fewer down to one (16 ragged sequences: 178 us with four heads,
    // 159 with two, 225 with one; 512 prompt tokens: 36, 42 and more)
    uint32_t heads = std::min(4u, group);
    while (heads > 1 && (uint64_t)m * n_kv_heads * (group / heads) * (head_dim / 64) < 4 * kAttnSimds) heads /= 2;
    const uint32_t waves_set = head_dim / 64, per_item = 4 / waves_set;  // waves per row set; row sets per item
    const uint32_t per = group / heads;  // row sets per token and KV head
    for (auto &q : seqs)
        for (uint32_t u = 0; u < n_kv_heads; u++, gid++) {
            const uint32_t sets = (q.second - q.first) * per;
            for (uint32_t r = 0; r < sets; r += per_item) {
                const uint32_t nt = std::min(per_item, sets - r), p1 = tok[q.first + (r + nt - 1) / per].pos + 1;
                items.push_back({q.first, nt, r, p1, u, 0});
                work.push_back((uint64_t)nt * p1);
                gids.push_back(gid);
            }
        }
    attn_place(items, work, gids, sv);
    return heads;
}

// Waves per row: one where a batch has rows enough to fill the chip, four
// for few rows of more than 1024 positions.  The line is where the four-wave
// workgroups (1024 threads, four rows) no longer all fit at once, two to a CU:
// us with one wave and with four, at 640 / 1920 / 2080 / 5120 rows of 1100
// positions 11 and 10 / 13.0 and 12.8 / 14 and 18.5 / 25 and 28; of 3000
// 24 and 18 / 28 and 23 / 29 and 35 / 55 and 54; of 3850 30 and 22 / 35 and 28 /
// 36 and 44 / 68 and 68.  Both numbers are the batch's, its longest row's and
// the rows of all: one row of 3900 positions among short ones is taken as
// if all were long, 2560 such rows 29 where four waves would take 21.
wm_attn_softmax_plan wm_attn_rows_softmax_plan(uint32_t n_rows, uint32_t n_max) {
    wm_attn_softmax_plan p{n_max <= 1024 || n_rows > 8 * kGemmCus ? 1u : 4u, 1u};
    while (256 * p.waves * p.slots < n_max) p.slots *= 2;
    return p;
}

void wm_launch_attn_rows(const float *q, const wm_batch_tok *tok, uint32_t m, uint32_t n_max,
                         uint32_t layer, uint32_t n_kv_heads, uint32_t head_dim, uint32_t group,
                         float scale, float *scores, float *out, uint32_t n_sc, uint32_t n_sv,
                         uint32_t sv_heads, hipStream_t s) {
    const uint32_t n_heads = n_kv_heads * group;
    uint8_t *base = reinterpret_cast<uint8_t *>(scores);
    uint8_t *live = base + attn_scores_part(m, n_heads, n_max);
    const wm_attn_item *items = wm_attn_rows_items(scores, m, n_heads, n_max);
    attn_rows_args a{q, tok, scores, out, layer, n_kv_heads * head_dim, n_heads,
                     attn_stride(n_max), n_max, scale, live, items, items + n_sc};
    const dim3 sgrid(n_sc);
#define WM_SCORES_CASE(HD, G)                                                                  \
    if (head_dim == HD && group == G)                                                          \
        hipLaunchKernelGGL((k_attn_scores_rows<HD, G>), sgrid, dim3(kScoreThreads), 0, s, a);
    WM_SCORES_CASE(128, 1) WM_SCORES_CASE(128, 2) WM_SCORES_CASE(128, 4) WM_SCORES_CASE(128, 8)
    WM_SCORES_CASE(64, 1) WM_SCORES_CASE(64, 2) WM_SCORES_CASE(64, 4) WM_SCORES_CASE(64, 8)
#undef WM_SCORES_CASE
    const uint32_t n_rows = m * n_heads;
    const wm_attn_softmax_plan sp = wm_attn_rows_softmax_plan(n_rows, n_max);
    const dim3 sm_grid((n_rows + kSmRows - 1) / kSmRows);
#define WM_SM_CASE(W, F)                                                                       \
    if (sp.waves == W && sp.slots == F)                                                        \
        hipLaunchKernelGGL((k_attn_softmax_rows<W, F>), sm_grid, dim3(kSmRows * W * 64), 0, s, a, n_rows);
    WM_SM_CASE(1, 1) WM_SM_CASE(1, 2) WM_SM_CASE(1, 4) WM_SM_CASE(1, 8) WM_SM_CASE(1, 16)
    WM_SM_CASE(4, 2) WM_SM_CASE(4, 4)
#undef WM_SM_CASE
#define WM_SV_CASE(HD, C)                                                                      \
    if (head_dim == HD && sv_heads == C)                                           \
        hipLaunchKernelGGL((k_attn_sv_rows<HD, C>), dim3(n_sv), dim3(256), 0, s, a, group);
    WM_SV_CASE(128, 1) WM_SV_CASE(128, 2) WM_SV_CASE(128, 4)
    WM_SV_CASE(64, 1) WM_SV_CASE(64, 2) WM_SV_CASE(64, 4)
#undef WM_SV_CASE
}
