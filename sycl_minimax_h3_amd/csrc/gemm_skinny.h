// gemm_skinny.h - the float linear with few rows on one side (h3s_linear, linear.hip): a text prompt's tokens against a
// layer's weights, or a sequence against the few rows of a LoRA's first factor. The long operand (L: the weights, or the
// tokens) is nearly all of the bytes, so such a product is bound by how fast L streams in, and then by the launch: where
// gemm_impl.h's 256 x 256 tiles give 21 tiles to 5376 rows of weights (168 blocks after the split along K, with partial
// sums of 256 padded rows each), a block here takes 64 or 128 rows of L against all rows of the short operand (S, up to
// 256 a block), and holds three to eight stages of both in flight.
// A CU's direct loads arrive at 52-61 bytes a nanosecond here (14336 -> 5376 in one part of 84 blocks: 137, 200 and 256 rows
// 110, 140 and 150 us) whatever the stages or the products beside them (a copy of the kernel without its LDS reads and
// products ran at the same speed), so the time of a block is its rows times its steps, and the launch weighs that against
// the partial sums (linear.hip, skinny_plan); the matrix cores are busy 17 % at 137 rows. Products with the next
// step's reads between them, and S's lines loaded ahead into the XCD's L2, gave nothing.
// bfloat16, 137 rows (cold weights): 5376 -> 5376 32.0 -> 24.3 us (16 rows: 25.8 -> 15.7; at 5 TB/s the weights take 11.6),
// 14336 -> 5376 59.3 -> 43.4; 512 rows 5376 -> 14336 107 -> 86 us; a LoRA's first factor 7168 -> 64 at 2159 tokens 29.8 ->
// 13.5, at 16896 78 -> 58, at 47104 182 -> 136 us.
//
// Block: eight wavefronts, 2 x 2 over the tile (each 32 MT rows of S x 32 of L) and two along K (each takes two of a
// step's four 32-byte slices: half the fragment reads a wavefront, and two wavefronts a SIMD; the second group's
// accumulators are added to the first's through LDS at the end). K advances 128 bytes a step through NS LDS stages filled
// by direct loads; stage kt is refilled right after the barrier that publishes stage kt + 1, whose fragments are read
// before kt's products. Tile, swizzle and fragments as in gemm_impl.h (gemm_unit).
// Loads past the matrices' ends, and of the steps past a part's last one, read zeros (buffer resources), so every step
// waits for the same number of loads.
// With parts > 1 each tile's K steps are shared by `parts` blocks that leave float32 sums in scratch (part-major); the
// merge kernel adds them in part order, then the bias, and rounds once.
#pragma once

#include "gemm_impl.h"

namespace h3 {

constexpr int kSkinnyThreads = 512;
// a block takes 64 MT rows of S and 64 NT of L; stages: as many as 160 KB hold, at most 8
constexpr int skinny_stage_bytes(int mt, int nt) { return 64 * (mt + nt) * kGemmBK; }
constexpr int skinny_stages(int mt, int nt) { return 160 * 1024 / skinny_stage_bytes(mt, nt) < 8 ? 160 * 1024 / skinny_stage_bytes(mt, nt) : 8; }
constexpr int skinny_per_cu(int mt, int nt) { return mt + nt == 2 ? 2 : 1; }    // blocks a CU (the smallest tile: two)

struct SkinnyArgs {
    const int8_t *s, *l;      // the short and the long operand's rows, kb bytes each
    int64_t S, L, kb;         // their rows; bytes a row
    const float* bias;        // [columns of out] or NULL
    void* out;                // [S, L], or [L, S] (SWAP: out's rows are L's)
    int out_dt;
    int ts, tl;               // tiles along S and L
    int parts;                // blocks that share a tile's K steps
    float* part;              // [tile, part, 64 MT * 64 NT] sums (parts > 1)
};

// one direct load of 16 bytes a lane through a buffer resource, as inline asm: see attn_dma16 (the compiler would make
// every LDS read wait for all direct loads in flight; wait_vm before each barrier orders these)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void skinny_dma16(const v4i& rsrc, uint32_t off, uint32_t lds_dst) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(off), "s"(rsrc), "s"(lds_dst) : "memory", "m0");
}
#pragma clang diagnostic pop
// a workgroup barrier after which every wavefront's LDS reads are done and all but its last N direct loads have landed
template <int N> __device__ __forceinline__ void skinny_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}
// the resource over `rows` rows of kb bytes from byte k0 of each on (live false: every load reads zeros)
__device__ __forceinline__ v4i skinny_rsrc(const int8_t* base, int64_t rows, int64_t kb, int64_t k0, bool live) {
    const uint64_t a = (uint64_t) (uintptr_t) (base + k0);
    const int64_t n = live ? rows * kb - k0 : 0;
    v4i r;
    r[0] = __builtin_amdgcn_readfirstlane((int) (uint32_t) a);
    r[1] = __builtin_amdgcn_readfirstlane((int) (uint32_t) (a >> 32) & 0xFFFF);
    r[2] = __builtin_amdgcn_readfirstlane((int) (uint32_t) (n < 0xFFFFFFFFll ? n : 0xFFFFFFFFll));
    r[3] = 0x00020000;
    return r;
}

// out[m][n .. n + 3] = v + bias, rounded to out's type; columns past N are not stored
__device__ __forceinline__ void skinny_store4(void* out, int out_dt, const float* bias, int64_t m, int64_t n, int64_t N, float4 v) {
    float x[4] = {v.x, v.y, v.z, v.w};
    const int64_t at = m * N + n;
    if (n + 3 < N && N % 4 == 0) {
        // (n is a multiple of 4 and out 16-byte aligned: whole 8- or 16-byte stores)
        if (bias)
#pragma unroll
            for (int q = 0; q < 4; ++q) x[q] = x[q] + bias[n + q];
        if (out_dt == H3S_F32) *reinterpret_cast<float4*>(reinterpret_cast<float*>(out) + at) = make_float4(x[0], x[1], x[2], x[3]);
        else
            *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(out) + at) =
                out_dt == H3S_BF16 ? make_uint2(pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3])) : make_uint2(pack_f16(x[0], x[1]), pack_f16(x[2], x[3]));
        return;
    }
    for (int q = 0; q < 4 && n + q < N; ++q) {
        const float y = bias ? x[q] + bias[n + q] : x[q];
        if (out_dt == H3S_F32) reinterpret_cast<float*>(out)[at + q] = y;
        else reinterpret_cast<uint16_t*>(out)[at + q] = (uint16_t) (out_dt == H3S_BF16 ? pack_bf16(y, 0.0f) : pack_f16(y, 0.0f));
    }
}
// where group g (four consecutive accumulator registers) of S fragment i and L fragment j lies in out, for the wavefront (ws, wl) of a tile
template <int MT, int NT, bool SWAP>
__device__ __forceinline__ void skinny_at(int64_t s0, int64_t l0, int ws, int wl, int i, int j, int g, int lane, int64_t* m, int64_t* n) {
    const int64_t s = s0 + ws * 32 * MT + 32 * i, l = l0 + wl * 32 * NT + 32 * j;
    const int reg = 8 * g + 4 * (lane >> 5), col = lane & 31;
    *m = SWAP ? l + col : s + col;
    *n = SWAP ? s + reg : l + reg;
}

template <int OP, int MT, int NT, bool SWAP>
__global__ __launch_bounds__(kSkinnyThreads, 2 * skinny_per_cu(MT, NT)) void gemm_skinny_kernel(SkinnyArgs P) {
    static_assert(OP == GEMM_BF16 || OP == GEMM_F16, "gemm_skinny_kernel: 16-bit operands");
    constexpr int NS = skinny_stages(MT, NT) / skinny_per_cu(MT, NT), STAGE = skinny_stage_bytes(MT, NT), LPW = MT + NT;
    constexpr int BS = 64 * MT, BL = 64 * NT, MAXT = MT > NT ? MT : NT;
    static_assert(NS >= 3 && NS * STAGE <= 160 * 1024 && NS * STAGE >= MT * NT * 16 * 1024, "gemm_skinny_kernel: LDS");
    __shared__ __attribute__((aligned(16))) int8_t lds[NS * STAGE];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave >> 2, ws = (wave >> 1) & 1, wl = wave & 1;
    const int64_t kb = P.kb;
    const int nk = (int) ((kb + kGemmBK - 1) / kGemmBK), tiles = P.ts * P.tl;
    // part-major, each XCD a contiguous run: its blocks share S's K range, and the tiles along S a panel of L
    const int id = gemm_xcd_id((int) blockIdx.x, tiles * P.parts), part = id / tiles, tile = id % tiles;
    const int64_t s0 = (int64_t) (tile % P.ts) * BS, l0 = (int64_t) (tile / P.ts) * BL;
    const int k_first = (int) ((int64_t) part * nk / P.parts), k_end = (int) ((int64_t) (part + 1) * nk / P.parts);
    const bool half_last = kb % kGemmBK != 0 && k_end == nk;

    // load q of a wavefront fills rows 64 q + 8 wave + lane / 8 of S (q < MT), or 64 (q - MT) + .. of L: whole 128-byte rows
    const int r = 8 * wave + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    uint32_t vo[MAXT];
#pragma unroll
    for (int q = 0; q < MAXT; ++q) vo[q] = (uint32_t) ((uint64_t) (r + 64 * q) * kb + 16 * c);
    const uint32_t lds0 = (uint32_t) (uintptr_t) lds + 1024 * wave;
    auto issue = [&](int kt, int st) {
        const int64_t k0 = (int64_t) kt * kGemmBK;
        const bool live = kt < k_end;
        const v4i rs = skinny_rsrc(P.s + s0 * kb, P.S - s0, kb, k0, live), rl = skinny_rsrc(P.l + l0 * kb, P.L - l0, kb, k0, live);
        const uint32_t d = __builtin_amdgcn_readfirstlane((int) (lds0 + st * STAGE));
#pragma unroll
        for (int q = 0; q < MT; ++q) skinny_dma16(rs, vo[q], d + 8192 * q);
#pragma unroll
        for (int q = 0; q < NT; ++q) skinny_dma16(rl, vo[q], d + 8192 * (MT + q));
    };
    // fragment bases of this wavefront's two slices 2 kg and 2 kg + 1
    int off_s[2], off_l[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int ch = 2 * (2 * kg + u) + (lane >> 5);
        off_s[u] = gemm_unit(ws * 32 * MT + (lane & 31), ch) * 16;
        off_l[u] = BS * kGemmBK + gemm_unit(wl * 32 * NT + (lane & 31), ch) * 16;
    }
    auto read = [&](int st, v4i (&a)[2][MT], v4i (&b)[2][NT]) {
        const int8_t* p = lds + st * STAGE;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int j = 0; j < NT; ++j) b[u][j] = *reinterpret_cast<const v4i*>(p + off_l[u] + 4096 * j);
#pragma unroll
            for (int i = 0; i < MT; ++i) a[u][i] = *reinterpret_cast<const v4i*>(p + off_s[u] + 4096 * i);
        }
    };
    v16f acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = (v16f) 0.0f;
    auto products = [&](const v4i (&a)[2][MT], const v4i (&b)[2][NT]) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const v4i f = SWAP ? a[u][i] : b[u][j], g = SWAP ? b[u][j] : a[u][i];
                    v16f& o = acc[i][j];
                    if constexpr (OP == GEMM_BF16)
                        o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf_g, f), __builtin_bit_cast(v8bf_g, g), o, 0, 0, 0);
                    else
                        o = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h_g, f), __builtin_bit_cast(v8h_g, g), o, 0, 0, 0);
                }
    };
    int st = 0;                                                // the stage of step kt
    auto step = [&](int kt, const v4i (&a)[2][MT], const v4i (&b)[2][NT], v4i (&an)[2][MT], v4i (&bn)[2][NT]) {
        // this stage's fragments are in registers and the next stage has landed, both for every wavefront
        skinny_barrier<(NS - 2) * LPW>();
        issue(kt + NS, st);
        st = st + 1 < NS ? st + 1 : 0;
        read(st, an, bn);
        // (a half step's slices 2 and 3, the second group's, are not in the row)
        if (!(half_last && kt == k_end - 1 && kg == 1)) products(a, b);
    };
    for (int q = 0; q < NS; ++q) issue(k_first + q, q);
    v4i xa[2][MT], xb[2][NT], ya[2][MT], yb[2][NT];
    skinny_barrier<(NS - 1) * LPW>();
    read(0, xa, xb);
    int kt = k_first;
    for (; kt + 1 < k_end; kt += 2) {
        step(kt, xa, xb, ya, yb);
        step(kt + 1, ya, yb, xa, xb);
    }
    if (kt < k_end) step(kt, xa, xb, ya, yb);
    skinny_barrier<0>();                                       // the stages are done with: LDS is the groups' now

    // the second group's sums to the first: [wavefront of the group][i][j][g][lane] float4
    float4* ex = reinterpret_cast<float4*>(lds) + (wave & 3) * (MT * NT * 4 * 64) + lane;
    if (kg == 1) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const v16f& a = acc[i][j];
                    ex[((i * NT + j) * 4 + g) * 64] = make_float4(a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]);
                }
    }
    __syncthreads();
    if (kg == 1) return;
    const int64_t N = SWAP ? P.S : P.L, M = SWAP ? P.L : P.S;
    float4* dst = reinterpret_cast<float4*>(P.part) + ((size_t) tile * P.parts + part) * (BS * BL / 4) + wave * (MT * NT * 4 * 64) + lane;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const v16f& a = acc[i][j];
                const int at = ((i * NT + j) * 4 + g) * 64;
                const float4 o = ex[at];
                const float4 v = make_float4(a[4 * g] + o.x, a[4 * g + 1] + o.y, a[4 * g + 2] + o.z, a[4 * g + 3] + o.w);
                int64_t m, n;
                skinny_at<MT, NT, SWAP>(s0, l0, ws, wl, i, j, g, lane, &m, &n);
                if (m >= M || n >= N) continue;                // (the merge reads none of these)
                if (P.parts > 1) dst[at] = v;
                else skinny_store4(P.out, P.out_dt, P.bias, m, n, N, v);
            }
}

// a thread sums four values' parts in part order: 64 MT * 64 NT / 4 threads a tile
template <int MT, int NT, bool SWAP>
__global__ __launch_bounds__(256) void skinny_merge_kernel(SkinnyArgs P) {
    constexpr int PER = 64 * MT * 64 * NT / 4;
    const int64_t t = (int64_t) blockIdx.x * 256 + threadIdx.x;
    const int tile = (int) (t / PER), e = (int) (t % PER), lane = e & 63, f = (e >> 6) % (MT * NT * 4), wave = (e >> 6) / (MT * NT * 4);
    if (tile >= P.ts * P.tl) return;
    int64_t m, n;
    skinny_at<MT, NT, SWAP>((int64_t) (tile % P.ts) * 64 * MT, (int64_t) (tile / P.ts) * 64 * NT, wave >> 1, wave & 1, f / (4 * NT), f / 4 % NT,
                            f % 4, lane, &m, &n);
    const int64_t N = SWAP ? P.S : P.L, M = SWAP ? P.L : P.S;
    if (m >= M || n >= N) return;
    const float4* src = reinterpret_cast<const float4*>(P.part) + (size_t) tile * P.parts * PER + e;
    float4 v = src[0];
    for (int p = 1; p < P.parts; ++p) {
        const float4 o = src[(size_t) p * PER];
        v = make_float4(v.x + o.x, v.y + o.y, v.z + o.z, v.w + o.w);
    }
    skinny_store4(P.out, P.out_dt, P.bias, m, n, N, v);
}

}  // namespace h3
