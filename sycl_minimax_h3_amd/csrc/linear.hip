// linear.hip - the plain (float) linear layers of kernels/h3sycl.h:87-93: h3s_linear (out = x w^T + bias),
// h3s_linear_acc (out += x w^T + bias, a LoRA's second factor) and h3s_scale_rows (kernels/h3sycl.cpp:656-739).
// bfloat16 and half operands with K a multiple of 32 run on the matrix cores in gemm_impl.h's pipeline
// (gemm_f16_kernel), or gemm_skinny.h's where one side has few rows (not h3s_linear_acc): float32 accumulation, and the epilogue adds the bias (and the old output) in float32 and rounds
// once to the output type, as the reference's matmul post-ops do, with no intermediate in memory. Every other call
// (float32 operands, other K, unaligned rows) runs on rocBLAS (a plain library GEMM, float32 accumulation, on the
// context's stream) into a float32 scratch, a chunk of rows at a time, and the same epilogue as a kernel of its own.
#include <rocblas/rocblas.h>

#include "gemm_skinny.h"

namespace h3 {

void release_blas(Ctx* c) {
    if (c->blas) (void) rocblas_destroy_handle((rocblas_handle) c->blas);
    c->blas = nullptr;
}

static rocblas_handle blas_of(Ctx* c) {
    if (!c->blas) {
        rocblas_handle h = nullptr;
        count_alloc();
        if (rocblas_create_handle(&h) != rocblas_status_success) { set_error("rocBLAS: no handle"); return nullptr; }
        if (rocblas_set_stream(h, c->stream) != rocblas_status_success) {
            (void) rocblas_destroy_handle(h);
            set_error("rocBLAS: could not bind the context's stream");
            return nullptr;
        }
        c->blas = h;
    }
    return (rocblas_handle) c->blas;
}

static rocblas_datatype blas_type(int dt) {
    return dt == H3S_F32 ? rocblas_datatype_f32_r : dt == H3S_F16 ? rocblas_datatype_f16_r : rocblas_datatype_bf16_r;
}

template <int DT> __device__ __forceinline__ float lin_load(const void* p, int64_t i) {
    if constexpr (DT == H3S_F32) return ((const float*) p)[i];
    else if constexpr (DT == H3S_BF16) return bf16_lo(((const uint16_t*) p)[i]);
    else return f16_lo(((const uint16_t*) p)[i]);
}
template <int DT> __device__ __forceinline__ void lin_store(void* p, int64_t i, float v) {
    if constexpr (DT == H3S_F32) ((float*) p)[i] = v;
    else if constexpr (DT == H3S_BF16) ((uint16_t*) p)[i] = (uint16_t) pack_bf16(v, 0.0f);
    else ((uint16_t*) p)[i] = (uint16_t) pack_f16(v, 0.0f);
}

// out[r, n] = round(acc[r, n] [+ bias[n]] [+ out[r, n]]) over rows [0, M)
template <int DT, bool ACC>
__global__ __launch_bounds__(256) void lin_epilogue_kernel(const float* __restrict__ acc, int64_t M, int64_t N,
                                                           const float* __restrict__ bias, void* out) {
    const int64_t n = M * N;
    for (int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t) gridDim.x * 256) {
        float v = acc[i];
        if (bias) v = v + bias[i % N];
        if constexpr (ACC) v = v + lin_load<DT>(out, i);
        lin_store<DT>(out, i, v);
    }
}

template <int DT>
__global__ __launch_bounds__(256) void scale_rows_kernel(void* x, int64_t M, int64_t C, const float* __restrict__ s) {
    const int64_t n = M * C;
    for (int64_t i = (int64_t) blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t) gridDim.x * 256)
        lin_store<DT>(x, i, lin_load<DT>(x, i) * s[i / C]);
}

static unsigned grid_of(int64_t n, const Ctx& c) {
    const int64_t b = (n + 255) / 256, cap = (int64_t) c.cus * 16;
    return (unsigned) (b < cap ? (b > 0 ? b : 1) : cap);
}

template <bool ACC>
static int launch_epilogue(Ctx* c, const float* acc, int64_t M, int64_t N, const float* bias, void* out, int out_dt) {
    const unsigned g = grid_of(M * N, *c);
    switch (out_dt) {
        case H3S_F32: lin_epilogue_kernel<H3S_F32, ACC><<<g, 256, 0, c->stream>>>(acc, M, N, bias, out); break;
        case H3S_F16: lin_epilogue_kernel<H3S_F16, ACC><<<g, 256, 0, c->stream>>>(acc, M, N, bias, out); break;
        default: lin_epilogue_kernel<H3S_BF16, ACC><<<g, 256, 0, c->stream>>>(acc, M, N, bias, out); break;
    }
    return 0;
}

// whether gemm_f16_kernel takes the product: 16-bit operands whose rows are whole 64-byte units (the pipeline's
// half K step) and start on 16-byte boundaries (out too), K * 2 below 2^24 bytes, tile counts within 32 bits
static bool mfma_takes(int dt, const void* x, const void* w, const void* out, int64_t M, int64_t K, int64_t N) {
    const int64_t tm = (M + kGemmBM - 1) / kGemmBM, tn = (N + kGemmBN - 1) / kGemmBN;
    return (dt == H3S_BF16 || dt == H3S_F16) && K % 32 == 0 && 2 * K < ((int64_t) 1 << 24) && aligned16(x) &&
           aligned16(w) && aligned16(out) && tm * tn <= 0x7fffffff;
}
// the merge of the split last tiles for operand type OP (out_dt: the output type; ACC: h3s_linear_acc, out in dt)
template <int OP, bool ACC>
static void merge_f16(Ctx* c, const GemmArgs& P, unsigned mgrid) {
    const bool b = P.bias != nullptr;
    if (P.out_dt == H3S_BF16) {
        if (b) gemm_merge_kernel<OP, H3S_ACT_NONE, false, ACC, H3S_BF16, true><<<mgrid, 256, 0, c->stream>>>(P);
        else gemm_merge_kernel<OP, H3S_ACT_NONE, false, ACC, H3S_BF16, false><<<mgrid, 256, 0, c->stream>>>(P);
    } else if (P.out_dt == H3S_F16) {
        if (b) gemm_merge_kernel<OP, H3S_ACT_NONE, false, ACC, H3S_F16, true><<<mgrid, 256, 0, c->stream>>>(P);
        else gemm_merge_kernel<OP, H3S_ACT_NONE, false, ACC, H3S_F16, false><<<mgrid, 256, 0, c->stream>>>(P);
    } else if constexpr (!ACC) {
        if (b) gemm_merge_kernel<OP, H3S_ACT_NONE, false, false, H3S_F32, true><<<mgrid, 256, 0, c->stream>>>(P);
        else gemm_merge_kernel<OP, H3S_ACT_NONE, false, false, H3S_F32, false><<<mgrid, 256, 0, c->stream>>>(P);
    }
}
static int linear_mfma(Ctx* c, const char* fn, const void* x, int dt, int64_t M, int64_t K, const void* w, int64_t N,
                       const float* bias, void* out, int out_dt, bool acc) {
    const int64_t tn = (N + kGemmBN - 1) / kGemmBN, kb = 2 * K;
    GemmPlan plan{4, 0, 1, 0.0};
    if (acc) {
        const int64_t tiles = (M + kGemmBM - 1) / kGemmBM * tn;
        plan.main_tiles = (int) tiles;
        gemm_plan_split(tiles, (kb + kGemmBK - 1) / kGemmBK, c->cus, &plan.main_tiles, &plan.split);
    } else {
        plan = gemm_plan(M, N, (kb + kGemmBK - 1) / kGemmBK, c->cus, true);
    }
    const int wi = plan.wi, main_tiles = plan.main_tiles, split = plan.split;
    const int64_t tm = (M + 64 * wi - 1) / (64 * wi);
    const int64_t tail = tm * tn - main_tiles;
    void* part = nullptr;
    if (split > 1) {
        part = c->scratch<float>(Ctx::GEMM_PART, (size_t) (tail * split) * kGemmTileAcc);
        if (!part) return -1;
    }
    const GemmArgs P{(const int8_t*) x, nullptr, M, kb, (const int8_t*) w, N, nullptr, bias, out, out_dt, (int) tm, (int) tn,
                     kb >= 12288 ? 4 : 8, main_tiles, split, part};
    const unsigned grid = (unsigned) (main_tiles + tail * split), mgrid = (unsigned) (tail * kGemmMergeBlocks);
    if (dt == H3S_BF16) {
        if (acc) gemm_f16_kernel<GEMM_BF16, true, 4><<<grid, kGemmThreads, 0, c->stream>>>(P);
        else if (wi == 2) gemm_f16_kernel<GEMM_BF16, false, 2><<<grid, kGemmThreads, 0, c->stream>>>(P);
        else if (wi == 3) gemm_f16_kernel<GEMM_BF16, false, 3><<<grid, kGemmThreads, 0, c->stream>>>(P);
        else gemm_f16_kernel<GEMM_BF16, false, 4><<<grid, kGemmThreads, 0, c->stream>>>(P);
        if (split > 1) { if (acc) merge_f16<GEMM_BF16, true>(c, P, mgrid); else merge_f16<GEMM_BF16, false>(c, P, mgrid); }
    } else {
        if (acc) gemm_f16_kernel<GEMM_F16, true, 4><<<grid, kGemmThreads, 0, c->stream>>>(P);
        else if (wi == 2) gemm_f16_kernel<GEMM_F16, false, 2><<<grid, kGemmThreads, 0, c->stream>>>(P);
        else if (wi == 3) gemm_f16_kernel<GEMM_F16, false, 3><<<grid, kGemmThreads, 0, c->stream>>>(P);
        else gemm_f16_kernel<GEMM_F16, false, 4><<<grid, kGemmThreads, 0, c->stream>>>(P);
        if (split > 1) { if (acc) merge_f16<GEMM_F16, true>(c, P, mgrid); else merge_f16<GEMM_F16, false>(c, P, mgrid); }
    }
    return launched(fn);
}

template <int OP, int MT, int NT, bool SWAP>
static void skinny_one(Ctx* c, const SkinnyArgs& P) {
    const int64_t tiles = (int64_t) P.ts * P.tl;
    gemm_skinny_kernel<OP, MT, NT, SWAP><<<(unsigned) (tiles * P.parts), kSkinnyThreads, 0, c->stream>>>(P);
    if (P.parts > 1) skinny_merge_kernel<MT, NT, SWAP><<<(unsigned) (tiles * (64 * MT * 64 * NT / 4 / 256)), 256, 0, c->stream>>>(P);
}
template <int OP, bool SWAP>
static void skinny_mt(Ctx* c, const SkinnyArgs& P, int mt, int nt) {
#define H3_SK(MM) { if (nt == 2) skinny_one<OP, MM, 2, SWAP>(c, P); else skinny_one<OP, MM, 1, SWAP>(c, P); }
    if (mt == 1) H3_SK(1)
    else if (SWAP || mt == 2) H3_SK(2)                           // (swapped: at most 128 rows of w)
    else if constexpr (!SWAP) {
        if (mt == 3) H3_SK(3)
        else H3_SK(4)
    }
#undef H3_SK
}
// The tile (64 mt rows of S, 64 nt of L) and the parts along K of an S x L product of nk K steps, by the least estimated
// time in microseconds (measured over S = 16 .. 512 rows against the DiT's layers and L = 300 .. 47104 rows against 16 ..
// 128, the choice is within 10 % of the fastest of all tiles and parts): a CU takes about 2.4 ns a row and step and at
// least 250 ns a step, the blocks run in rounds of one a CU, memory gives about 5 TB/s (7 for what the 256 MB cache beside
// it may hold), and parts cost their float32 sums written and read once and the merge's launch.
struct SkinnyPlan { int mt, nt, parts; int64_t blocks, rows; double us; };
static SkinnyPlan skinny_plan(int64_t S, int64_t L, int64_t nk, int cus) {
    SkinnyPlan best{0, 0, 0, 0, 0, 1e300};
    const int64_t ts = (S + 255) / 256;
    const int mt = (int) ((S + 64 * ts - 1) / (64 * ts));
    const int64_t rows = (S + ts - 1) / ts;
    for (int nt = 1; nt <= 2; ++nt)
        for (int parts = 1; parts <= 8; ++parts) {
            if (parts > 1 && 4 * parts > nk) break;              // at least 4 steps a part
            const int64_t blocks = ts * ((L + 64 * nt - 1) / (64 * nt)) * parts;
            const double run = (double) ((blocks + cus - 1) / cus) * (double) ((nk + parts - 1) / parts) *
                               std::max(0.25, 0.0024 * (double) (rows + 64 * nt));
            const double bytes = (double) (S + L) * (double) nk * kGemmBK, floor = bytes / (bytes > 256e6 ? 5e6 : 7e6);
            const double us = std::max(run, floor) + (parts > 1 ? 2.0 + (double) parts * (double) S * (double) L * 8 / 3.5e6 : 0.0);
            if (us < best.us) best = {mt, nt, parts, blocks, rows, us};
        }
    return best;
}
// Whether gemm_impl.h's tiles take a product that skinny_plan has planned (p) after all: not where its tiles are split in
// parts; where it takes several rounds of more than 64 rows, unless their loads alone take the time (an out of few columns: up
// to 16 steps); and else by the two whole times in microseconds. Here: 0.0026 a row and step, a block's end (the groups'
// exchange, 8-byte stores) 0.76 a 64 x 64 piece and round, 3.8 for the launch. There: gemm_plan's estimate, 3.9 for the
// launch with the short epilogue of a tile inside out, 0.035 more a live row of a tile cut at out's edge (its stores go
// element by element), 5.5 with a merge. Weights that a model's other layers have pushed out of the caches come slower there
// than here: a step of 256, 192 or 128 rows then takes 1.75, 1.55 or 1.33 however few the blocks (counted in full from 32
// steps, where the weights are megabytes, and half from 8). Operands past the 256 MB cache come at 6.5 TB/s here, by the
// blocks' share of the CUs, and at 5 there. Timed both ways over 1 .. 512 rows against 256 .. 65536 outputs, and 513 .. 47104
// against 8 .. 128, of 64 .. 14336 features (bfloat16, 2099 products, their weights cached): the choice is 0.4 % off the faster
// on average, and within 5 % of it in 96 %; with cold weights (189 products) within 3 % of always taking this kernel where that
// is faster. Always here, products of one to four steps and of more outputs than fill one round had lost to the tiles: 512
// rows 64 -> 28672 8.5 -> 24.1 us, 512 rows 5376 -> 28672 143 -> 181, 256 rows 64 -> 5376 5.7 -> 7.9.
static bool skinny_loses(const SkinnyPlan& p, bool swap, int64_t M, int64_t N, int64_t nk, int cus) {
    if (p.parts > 1) return false;
    const int64_t round = (int64_t) cus * skinny_per_cu(p.mt, p.nt), rounds = (p.blocks + round - 1) / round;
    const double bytes = (double) (M + N) * (double) nk * kGemmBK;
    const bool cached = bytes <= 256e6;
    const double run = (double) ((p.blocks + cus - 1) / cus * nk) * std::max(0.25, 0.0026 * (double) (p.rows + 64 * p.nt));
    const double from = cached ? bytes / 7e6 : bytes / (6.5e6 * std::min(1.0, (double) p.blocks / cus));
    const bool by_loads = p.us <= 1.0001 * bytes / (cached ? 7e6 : 5e6);
    if (rounds > 1 && p.rows > 64 && (swap ? nk <= 16 : M > 256 || !by_loads)) return true;
    const GemmPlan g = gemm_plan(M, N, nk, cus, true);
    const int64_t bm = 64 * g.wi, tm = (M + bm - 1) / bm, tn = (N + kGemmBN - 1) / kGemmBN;
    double tiles = g.us;
    if (!cached || nk >= 8) {
        const double step = g.wi == 4 ? 1.75 : g.wi == 3 ? 1.55 : 1.33;
        double t = (double) ((g.main_tiles + cus - 1) / cus * nk) * step;
        if (g.split > 1)
            t += (double) ((nk + g.split - 1) / g.split) * step +
                 0.1 * (double) ((tm * tn - g.main_tiles) * g.split) * std::min(1.0, (double) M / kGemmBM);
        if (cached && nk < 32) t = 0.5 * (t + tiles);
        tiles = std::max({tiles, t, cached ? 0.0 : bytes / 5e6});
    }
    int64_t cut = 0;                                             // live rows that cut tiles store one after the other
    if (g.split == 1) {
        cut = M % bm * ((tn + cus - 1) / cus);
        if (N % kGemmBN) cut = std::max(cut, std::min(M, bm) * ((tm + cus - 1) / cus));
    }
    const double here = 3.8 + 0.76 * (double) (p.mt * p.nt * rounds) + std::max(run, from);
    const double there = 3.9 + 0.035 * (double) cut + (g.split > 1 ? 5.5 : 0.0) + tiles;
    return there < here;
}
// h3s_linear with few rows on one side (gemm_skinny.h): at most 512 rows of x, or at most 128 of w. Above, gemm_impl.h's
// tiles have the rows to fill them (768 rows 5376 -> 5376: 65 against 66 us at the best tile here; 256 rows of w at 16896
// tokens 95 against 137). 1: not a product it takes.
static int linear_skinny(Ctx* c, const char* fn, const void* x, int dt, int64_t M, int64_t K, const void* w, int64_t N,
                         const float* bias, void* out, int out_dt) {
    const int64_t kb = 2 * K, nk = (kb + kGemmBK - 1) / kGemmBK;
    SkinnyPlan p{0, 0, 0, 0, 0, 1e300};
    bool swap = false;
    if (M <= 512) p = skinny_plan(M, N, nk, c->cus);
    if (N <= 128) {
        const SkinnyPlan q = skinny_plan(N, M, nk, c->cus);
        if (q.us < p.us) { p = q; swap = true; }
    }
    if (!p.mt || skinny_loses(p, swap, M, N, nk, c->cus)) return 1;
    const int64_t S = swap ? N : M, L = swap ? M : N;
    const int64_t ts = (S + 64 * p.mt - 1) / (64 * p.mt), tl = (L + 64 * p.nt - 1) / (64 * p.nt);
    if (ts * tl * 64 > 0x7fffffff) return 1;                     // (blocks, and the merge's, within 32 bits)
    SkinnyArgs P{(const int8_t*) (swap ? w : x), (const int8_t*) (swap ? x : w), S, L, kb, bias, out, out_dt, (int) ts, (int) tl, p.parts, nullptr};
    // (no room for the partial sums under the memory cap: each tile whole)
    if (P.parts > 1 && !(P.part = c->scratch<float>(Ctx::GEMM_PART, (size_t) (ts * tl * P.parts) * (64 * p.mt * 64 * p.nt)))) P.parts = 1;
    if (dt == H3S_BF16) { if (swap) skinny_mt<GEMM_BF16, true>(c, P, p.mt, p.nt); else skinny_mt<GEMM_BF16, false>(c, P, p.mt, p.nt); }
    else { if (swap) skinny_mt<GEMM_F16, true>(c, P, p.mt, p.nt); else skinny_mt<GEMM_F16, false>(c, P, p.mt, p.nt); }
    return launched(fn);
}

// the product x [M, K] . w^T (w [N, K]), both in dt, into out (or out +=): on the matrix cores, or on rocBLAS a
// chunk of rows at a time
static int linear(Ctx* c, const char* fn, const void* x, int dt, int64_t M, int64_t K, const void* w, int64_t N,
                  const float* bias, void* out, int out_dt, bool acc) {
    if (K > 0x7fffffff || N > 0x7fffffff) return fail(std::string(fn) + ": K and N must be below 2^31");
    if (mfma_takes(dt, x, w, out, M, K, N)) {
        const int r = acc ? 1 : linear_skinny(c, fn, x, dt, M, K, w, N, bias, out, out_dt);
        return r != 1 ? r : linear_mfma(c, fn, x, dt, M, K, w, N, bias, out, out_dt, acc);
    }
    rocblas_handle h = blas_of(c);
    if (!h) return -1;
    // rows a chunk: the float32 product of a chunk takes at most 256 MiB (and at most 8192 rows, as the reference)
    int64_t rows = (int64_t) (256 << 20) / (N * 4);
    rows = rows < 1 ? 1 : rows > 8192 ? 8192 : rows;
    rows = rows < M ? rows : M;
    float* tmp = c->scratch<float>(Ctx::LIN_F32, (size_t) (rows * N));
    if (!tmp) return -1;
    const size_t xe = (size_t) elem_size(dt), oe = (size_t) elem_size(out_dt);
    const float one = 1.0f, zero = 0.0f;
    for (int64_t r0 = 0; r0 < M; r0 += rows) {
        const int64_t m = M - r0 < rows ? M - r0 : rows;
        // column-major view: tmp^T [N, m] = w [N, K] (stored as K x N, transposed) . x^T [K, m]
        const rocblas_status st = rocblas_gemm_ex(h, rocblas_operation_transpose, rocblas_operation_none, (rocblas_int) N,
                                                  (rocblas_int) m, (rocblas_int) K, &one, w, blas_type(dt), (rocblas_int) K,
                                                  (const char*) x + (size_t) (r0 * K) * xe, blas_type(dt), (rocblas_int) K,
                                                  &zero, tmp, rocblas_datatype_f32_r, (rocblas_int) N, tmp,
                                                  rocblas_datatype_f32_r, (rocblas_int) N, rocblas_datatype_f32_r,
                                                  rocblas_gemm_algo_standard, 0, 0);
        if (st != rocblas_status_success)
            return fail(std::string(fn) + ": rocBLAS gemm_ex failed (" + rocblas_status_to_string(st) + ")");
        char* o = (char*) out + (size_t) (r0 * N) * oe;
        if (acc) launch_epilogue<true>(c, tmp, m, N, bias, o, out_dt);
        else launch_epilogue<false>(c, tmp, m, N, bias, o, out_dt);
        if (launched(fn)) return -1;
    }
    return 0;
}

}  // namespace h3

using namespace h3;

H3S_EXPORT int h3s_linear(void* ctx, const void* x, int dt, int64_t M, int64_t K, const void* w, int64_t N, const float* bias,
                          void* out, int out_dt) try {
    const char* fn = "h3s_linear";
    if (M <= 0 || K <= 0 || N <= 0) return 0;
    if (!dt_ok(dt) || !dt_ok(out_dt)) return fail(std::string(fn) + ": unknown element type");
    if (!x || !w || !out) return fail(std::string(fn) + ": x, w and out are required");
    Ctx* c = ctx_of(ctx, fn);
    if (!c) return -1;
    return linear(c, fn, x, dt, M, K, w, N, bias, out, out_dt, false);
} catch (const std::exception& e) { return fail(e.what()); }

H3S_EXPORT int h3s_linear_acc(void* ctx, const void* x, int dt, int64_t M, int64_t K, const void* w, int64_t N,
                              const float* bias, void* out) try {
    const char* fn = "h3s_linear_acc";
    if (M <= 0 || K <= 0 || N <= 0) return 0;
    if (!dt_ok(dt)) return fail(std::string(fn) + ": unknown element type");
    if (!x || !w || !out) return fail(std::string(fn) + ": x, w and out are required");
    Ctx* c = ctx_of(ctx, fn);
    if (!c) return -1;
    return linear(c, fn, x, dt, M, K, w, N, bias, out, dt, true);
} catch (const std::exception& e) { return fail(e.what()); }

H3S_EXPORT int h3s_scale_rows(void* ctx, void* x, int dt, int64_t M, int64_t C, const float* s) try {
    const char* fn = "h3s_scale_rows";
    if (M <= 0 || C <= 0) return 0;
    if (!dt_ok(dt)) return fail(std::string(fn) + ": unknown element type");
    if (!x || !s) return fail(std::string(fn) + ": x and s are required");
    Ctx* c = ctx_of(ctx, fn);
    if (!c) return -1;
    const unsigned g = grid_of(M * C, *c);
    switch (dt) {
        case H3S_F32: scale_rows_kernel<H3S_F32><<<g, 256, 0, c->stream>>>(x, M, C, s); break;
        case H3S_F16: scale_rows_kernel<H3S_F16><<<g, 256, 0, c->stream>>>(x, M, C, s); break;
        default: scale_rows_kernel<H3S_BF16><<<g, 256, 0, c->stream>>>(x, M, C, s); break;
    }
    return launched(fn);
} catch (const std::exception& e) { return fail(e.what()); }
