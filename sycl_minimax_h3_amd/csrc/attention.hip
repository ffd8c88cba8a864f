// attention.hip - h3s_attention, h3s_attention_batch (kernels/h3sycl.h:185-197, kernels/h3sycl.cpp:1433-1917) and
// h3s_attention_causal (kernels/h3sycl.h:104-108) on the kernels of attn_impl.h. The form follows the reference's
// choice: the int8 (SageAttention) form for sequences of at least H3S_SAGE_MIN_S tokens (8192) with heads of 64 or
// 128 features unless H3S_ATTN=onednn (kernels/h3sycl.cpp:1706), the 16-bit form otherwise. Any head size up to 256
// (the causal form's limit, h3sycl.cpp:877): a head runs in the kernel of 64, 128 or 256 features, zero-padded past D.
#include <cmath>
#include <cstdio>

#include "attn_impl.h"

namespace h3 {

// q of Hq heads (row stride qs) and k, v of Hkv heads (row stride kvs) prepared into aq [Hq, Sp, DK], ak [Hkv, Sp, DK]
// (int8 codes with their scales for SAGE, else half) and av [Hkv, Sp / 32, DK, 32] (half), DK = attn_dk(D), zero past D
// (q_in_kernel: the attention kernel forms q's fragments from q itself, so q is not prepared)
template <int DT>
static void prep(Ctx* c, const void* q, const void* k, const void* v, int64_t S, int64_t Sp, int64_t Hq, int64_t Hkv, int D,
                 int64_t qs_stride, int64_t kv_stride, bool sage, bool q_in_kernel, int8_t* aq, int8_t* ak, uint16_t* av,
                 float* qs, float* ks, float* km) {
    const unsigned qblocks = (unsigned) (Hq * (Sp / kAttnRows)), kvblocks = (unsigned) (Hkv * (Sp / kAttnRows));
    const int DK = attn_dk(D);
    // 16-byte rows: every tensor aligned, the strides whole numbers of 16-byte vectors, and a head of exactly 64, 128
    // or 256 features (no padding)
    const bool vec = aligned16(q) && aligned16(k) && aligned16(v) && (qs_stride * elem_size(DT)) % 16 == 0 &&
                     (kv_stride * elem_size(DT)) % 16 == 0 && D == DK;
    auto qk = [&](const void* src, int64_t stride, unsigned blocks, const float* mean, int8_t* dst, float* sc) {
#define H3_QK(SG, DD) attn_qk_prep_vec_kernel<DT, SG, DD><<<blocks, 256, 0, c->stream>>>(src, S, Sp, stride, mean, dst, sc)
        if (!vec) {
            if (sage) attn_qk_prep_kernel<DT, true><<<blocks, 256, 0, c->stream>>>(src, S, Sp, D, DK, stride, mean, dst, sc);
            else attn_qk_prep_kernel<DT, false><<<blocks, 256, 0, c->stream>>>(src, S, Sp, D, DK, stride, mean, dst, sc);
        } else if (sage) {
            // (the int8 form is for heads of 64 or 128 features only)
            if (D == 128) H3_QK(true, 128);
            else H3_QK(true, 64);
        } else {
            if (D == 256) H3_QK(false, 256);
            else if (D == 128) H3_QK(false, 128);
            else H3_QK(false, 64);
        }
#undef H3_QK
    };
    // k and v: together where both take the 16-byte form
    auto kv = [&](const float* mean, float* sc) {
#define H3_KV(SG, DD) attn_kv_prep_vec_kernel<DT, SG, DD><<<2 * kvblocks, 256, 0, c->stream>>>(k, v, S, Sp, kv_stride, mean, ak, sc, av)
        if (!vec) {
            qk(k, kv_stride, kvblocks, mean, ak, sc);
            attn_v_prep_kernel<DT><<<kvblocks, 256, 0, c->stream>>>(v, S, Sp, D, __builtin_ctz((unsigned) DK), kv_stride, av);
        } else if (sage) {
            if (D == 128) H3_KV(true, 128);
            else H3_KV(true, 64);
        } else {
            if (D == 256) H3_KV(false, 256);
            else if (D == 128) H3_KV(false, 128);
            else H3_KV(false, 64);
        }
#undef H3_KV
    };
    if (sage) {
        // k's mean per (head, feature) of the D features; the 16-byte form takes 16 features a block, or 32 where 16
        // would make more blocks than the device runs at once
        const int64_t hd = Hkv * D;
        const bool wide = hd % kKmeanFeatWide == 0 && hd / kKmeanFeat > c->cus;
        if (vec && wide) attn_kmean_kernel<DT, kKmeanFeatWide><<<(unsigned) (hd / kKmeanFeatWide), 256, 0, c->stream>>>(k, S, kv_stride, km);
        else if (vec && hd % kKmeanFeat == 0) attn_kmean_kernel<DT, kKmeanFeat><<<(unsigned) (hd / kKmeanFeat), 256, 0, c->stream>>>(k, S, kv_stride, km);
        else attn_kmean_rows_kernel<DT><<<(unsigned) ((hd + 255) / 256), 256, 0, c->stream>>>(k, S, hd, kv_stride, km);
    }
    if (!q_in_kernel) qk(q, qs_stride, qblocks, nullptr, aq, sage ? qs : nullptr);
    kv(sage ? km : nullptr, sage ? ks : nullptr);
}

// Whether the causal form takes two key groups a block: where the launch's time is the walk of its longest blocks (few heads,
// long rows). bfloat16, heads of 128, one group a block -> two, all else alike: 8 heads 2048 tokens 48.9 -> 40.9 us, 32 heads
// 600 tokens 22.1 -> 20.5, 2048 tokens 61.7 -> 57.7; but 64 heads 600 tokens 23.7 -> 24.7, 2048 tokens 94.5 -> 103 (the
// blocks fill the device: there two blocks of one group a CU run without a common barrier), and 100 tokens 11.3 -> 12.4 (two
// tiles: nothing to share out)
static bool attn_causal_groups(int64_t L, int64_t Hq, int cus) { return L >= 512 && 8 * Hq <= cus; }
// Which of the wide kernel's n blocks of T key tiles run whole (the first `full`), and into how many blocks of `ts`
// consecutive tiles each of the others is split (`ns`, at most max_ns; 1: none): the least estimated time, in key tiles of a
// block that has its CU to itself. Two blocks that share a CU take 1.5 a tile each; a block's start and end cost 5 (1.7 where
// it is alone); a split costs the merge's launch (7) and every part 0.045 for its partial sums, 130 KiB written and read.
// Candidates: whole multiples of one or two blocks a CU stay whole, or none (at most two blocks a CU in all). After a round
// of two blocks a CU, the 16-bit form's next blocks do not spread one a CU: a last round of at most one a CU takes 1.2 there,
// and a whole block a CU with parts beside it is left to the first round. Parts are bounded by four a CU (133 MiB of scratch
// on 256 CUs). All choices timed at 1 .. 64 heads, 33 .. 16896 tokens: this takes the fastest, or one within 3 % of it, in 257 of 267
// cases, and the worst is 10 % off. Splitting whenever a last round filled at most half of two blocks a CU, into
// as many parts as fitted, lost where a part was short (56 heads: 64 tokens 21.7 -> 14.5 us, 137 tokens 31.7 -> 17.8, 600
// tokens 52.0 -> 38.7, 1000 tokens 69.9 -> 53.8) and left 257 .. 511 blocks whole (int8 form, 8300 tokens: 8 heads 375 -> 280
// us, 40 heads 1178 -> 1074; 16896 tokens 4 heads 749 -> 530).
struct AttnSplit { int64_t full; int ns, ts; };
static double attn_split_time(int64_t blocks, int64_t T, int64_t cus, double late) {
    const int64_t rounds = blocks / (2 * cus), rem = blocks % (2 * cus);
    return (double) rounds * (1.5 * (double) T + 5.0) +
           (rem == 0 ? 0.0 : rem <= cus ? (rounds ? late : 1.0) * (double) T + 1.7 : 1.5 * (double) T + 5.0);
}
static AttnSplit attn_split_plan(int64_t n, int64_t T, int64_t cus, int64_t max_ns, bool sage) {
    const double late = sage ? 1.0 : 1.2;
    AttnSplit best{n, 1, 0};
    double least = attn_split_time(n, T, cus, late);
    const int64_t fulls[3] = {0, n / cus * cus, n / (2 * cus) * (2 * cus)};
    for (const int64_t full : fulls) {
        const int64_t rest = n - full;
        const bool beside = full % (2 * cus) != 0;             // a whole block a CU, the parts in their CUs' second places
        if (rest == 0 || rest > 2 * cus || (beside && full > cus && !sage)) continue;
        for (int64_t want = 2; want <= max_ns && want <= T && rest * want <= 4 * cus; ++want) {
            const int64_t ts = (T + want - 1) / want, parts = rest * want;
            if ((T + ts - 1) / ts != want) continue;           // (a smaller count has the same longest part)
            double t = attn_split_time(full / (2 * cus) * (2 * cus), T, cus, late) + 7.0 + 0.045 * (double) parts;
            if (beside) {
                // u tiles beside the whole block, the rest of the longer of the two alone
                const double u = (double) ((parts + cus - 1) / cus) * ((double) ts + 5.0 / 1.5), w = (double) T;
                t += 1.7 + (u <= w ? 1.5 * u + (w - u) : 1.5 * w + (u - w));
            } else {
                // (parts of more than one round start unevenly)
                t += attn_split_time(parts, ts, cus, late) * (parts > 2 * cus ? 1.06 : 1.0);
            }
            if (t < least) { least = t; best = {full, (int) want, (int) ts}; }
        }
    }
    return best;
}

// one sequence: S query rows of Hq heads (row stride qs_stride) over S key/value rows of Hkv heads (kv_stride);
// causal: query i sees keys 0 .. i (the 16-bit form, as the reference's causal kernel computes in float)
static int attention_one(Ctx* c, const char* fn, const void* q, const void* k, const void* v, int dt, int64_t S, int64_t Hq,
                         int64_t Hkv, int64_t D, int64_t qs_stride, int64_t kv_stride, void* out, int out_dt, bool causal) {
    // the int8 form as the reference takes it (kernels/h3sycl.cpp:1706): heads of 64 or 128 features, and S * D * H
    // within int32; every other call runs the 16-bit form
    const bool sage = !causal && c->sage_want && S >= c->sage_min_s && (D == 64 || D == 128) && S <= INT32_MAX / D / Hq;
    // heads of 128 features into an aligned out, no causal mask: the wide kernel (256 queries a block)
    const bool pp = !causal && D == 128 && aligned16(out);
    const int64_t qblock = pp ? kAttnPPQ : kAttnQBlock;
    const int64_t Sp = (S + qblock - 1) / qblock * qblock, nbp = Sp / kAttnRows;
    const int64_t esz = sage ? 1 : 2, DK = attn_dk(D);
    if (Hq * (Sp / qblock) > 0x7fffffff) return fail(std::string(fn) + ": too many query blocks");
    // the wide kernel, and the 16-bit form of the others, read q's rows themselves where they are whole 16-byte vectors of
    // unpadded heads (no prepared q then: one launch less, and q neither written nor read again)
    // (a block writes its rows of out when it ends, where others have yet to read their rows of q: an out that overlaps q
    // otherwise than row on row has q prepared first. k and v are always prepared before any block runs.)
    const char *qb0 = (const char*) q, *ob0 = (const char*) out;
    const bool apart = ob0 + S * Hq * D * elem_size(out_dt) <= qb0 || qb0 + S * qs_stride * elem_size(dt) <= ob0 ||
                       (ob0 == qb0 && qs_stride == Hq * D && elem_size(dt) == elem_size(out_dt));
    const bool q_in_kernel = (pp || !sage) && apart && D == DK && aligned16(q) && (qs_stride * elem_size(dt)) % 16 == 0;
    int8_t* aq = q_in_kernel ? nullptr : c->scratch<int8_t>(Ctx::ATT_Q, (size_t) (Sp * Hq * DK * esz));
    const size_t over = pp ? kAttnOver : 0;                   // what its last direct loads read past the end
    int8_t* ak = c->scratch<int8_t>(Ctx::ATT_K, (size_t) (Sp * Hkv * DK * esz) + over);
    uint16_t* av = c->scratch<uint16_t>(Ctx::ATT_V, (size_t) (Sp * Hkv * DK) + over / 2);
    float* af = c->scratch<float>(Ctx::ATT_AUX, (size_t) ((Hq + Hkv) * nbp + Hkv * D));
    if ((!aq && !q_in_kernel) || !ak || !av || !af) return -1;
    float *qs = af, *ks = af + Hq * nbp, *km = af + (Hq + Hkv) * nbp;
    PhaseTimer timer(c);
    timer.mark();
    switch (dt) {
        case H3S_BF16: prep<H3S_BF16>(c, q, k, v, S, Sp, Hq, Hkv, (int) D, qs_stride, kv_stride, sage, q_in_kernel, aq, ak, av, qs, ks, km); break;
        case H3S_F16: prep<H3S_F16>(c, q, k, v, S, Sp, Hq, Hkv, (int) D, qs_stride, kv_stride, sage, q_in_kernel, aq, ak, av, qs, ks, km); break;
        default: prep<H3S_F32>(c, q, k, v, S, Sp, Hq, Hkv, (int) D, qs_stride, kv_stride, sage, q_in_kernel, aq, ak, av, qs, ks, km); break;
    }
    if (launched(fn)) return -1;
    AttnArgs P;
    P.q = aq; P.k = ak; P.vt = av; P.qs = qs; P.ks = ks;
    P.S = S; P.Sp = Sp; P.H = Hq;
    P.c = (float) (1.4426950408889634 * (double) (1.0f / std::sqrt((float) D)));
    P.out = out; P.out_dt = out_dt; P.D = (int) D;
    P.nqb = (int) (Sp / qblock);
    P.kvdiv = (int) (Hq / Hkv);
    P.Spk = Sp;
    P.qraw = q_in_kernel ? q : nullptr;
    P.qstride = qs_stride;
    P.q_dt = dt;
    const int64_t nblocks = Hq * P.nqb;
    P.nfull = nblocks; P.nsplit = 1; P.ts = 0; P.po = nullptr; P.pml = nullptr;
    // the wide kernel's blocks that are split along the keys (their results combined by attn_merge_kernel)
    int64_t tail = 0;
    if (pp) {
        const AttnSplit sp = attn_split_plan(nblocks, (S + kAttnVT - 1) / kAttnVT, c->cus, c->attn_split, sage);
        const int64_t last = nblocks - sp.full;
        // (no room for the partial sums under the memory cap: every block runs whole)
        if (sp.ns > 1 && (P.po = c->scratch<float>(Ctx::ATT_PART, (size_t) (last * sp.ns * kAttnPPQ * (128 + 2))))) {
            P.pml = P.po + last * sp.ns * kAttnPPQ * 128;
            tail = last;
            P.nfull = sp.full; P.nsplit = sp.ns; P.ts = sp.ts;
        }
    }
    const unsigned grid = (unsigned) (P.nfull + tail * P.nsplit);
    timer.mark();
    // heads of 64, 128 or 256 features into an aligned out take the plain stores; others the masked ones
    const bool pad = D != DK || !aligned16(out);
#define H3_ATTN_D(SG, DD, CA)                                                                  \
    {                                                                                          \
        if (pad) attn_kernel<SG, DD, CA, true><<<grid, 256, 0, c->stream>>>(P);               \
        else attn_kernel<SG, DD, CA, false><<<grid, 256, 0, c->stream>>>(P);                  \
    }
    if (pp) {
        if (sage) attn_pl_kernel<true, 6><<<grid, 256, 0, c->stream>>>(P);
        else attn_pl_kernel<false, 4><<<grid, 256, 0, c->stream>>>(P);
        if (tail) attn_merge_kernel<<<(unsigned) ((tail * kAttnPPQ * 32 + 255) / 256), 256, 0, c->stream>>>(P, tail);
    } else if (causal && DK <= 128 && attn_causal_groups(S, Hq, c->cus)) {
        if (DK == 128) { if (pad) attn_kernel<false, 128, true, true, 2><<<grid, 512, 0, c->stream>>>(P); else attn_kernel<false, 128, true, false, 2><<<grid, 512, 0, c->stream>>>(P); }
        else { if (pad) attn_kernel<false, 64, true, true, 2><<<grid, 512, 0, c->stream>>>(P); else attn_kernel<false, 64, true, false, 2><<<grid, 512, 0, c->stream>>>(P); }
    } else if (causal) {
        if (DK == 256) H3_ATTN_D(false, 256, true)
        else if (DK == 128) H3_ATTN_D(false, 128, true)
        else H3_ATTN_D(false, 64, true)
    } else if (DK == 128) {
        // (heads of 65 to 127 features, or an out off 16-byte boundaries: the others took the wide kernel)
        if (sage) attn_kernel<true, 128, false, true><<<grid, 256, 0, c->stream>>>(P);
        else attn_kernel<false, 128, false, true><<<grid, 256, 0, c->stream>>>(P);
    } else if (DK == 256) {
        H3_ATTN_D(false, 256, false)
    } else if (sage) {
        H3_ATTN_D(true, 64, false)
    } else {
        H3_ATTN_D(false, 64, false)
    }
#undef H3_ATTN_D
    if (launched(fn)) return -1;
    timer.mark();
    const std::vector<float> ms = timer.elapsed();
    if (ms.size() == 2)   // H3S_PROFILE (kernels/h3sycl.cpp:1753-1760)
        std::fprintf(stderr, "h3hip: attention (%s) S=%lld H=%lld D=%lld: preparation %.2f ms, attention %.2f ms\n",
                     sage ? "int8" : causal ? "16-bit, causal" : "16-bit", (long long) S, (long long) Hq, (long long) D, ms[0],
                     ms[1]);
    return 0;
}

static int attention_checks(const char* fn, int dt, int64_t H, int64_t D, int64_t stride, int out_dt, const void* q,
                            const void* k, const void* v, const void* out) {
    if (stride < H * D) return fail(std::string(fn) + ": the row stride is shorter than a row");
    if (!dt_ok(dt) || !dt_ok(out_dt)) return fail(std::string(fn) + ": unknown element type");
    if (D > kAttnMaxD) return fail(std::string(fn) + ": head size " + std::to_string(D) + " (at most 256)");
    if (!q || !k || !v || !out) return fail(std::string(fn) + ": q, k, v and out are required");
    return 0;
}

}  // namespace h3

using namespace h3;

H3S_EXPORT int h3s_attention(void* ctx, const void* q, const void* k, const void* v, int dt, int64_t S, int64_t H, int64_t D,
                             int64_t stride, void* out, int out_dt) try {
    const char* fn = "h3s_attention";
    if (S <= 0 || H <= 0 || D <= 0) return 0;
    if (attention_checks(fn, dt, H, D, stride, out_dt, q, k, v, out)) return -1;
    Ctx* c = ctx_of(ctx, fn);
    if (!c) return -1;
    return attention_one(c, fn, q, k, v, dt, S, H, H, D, stride, stride, out, out_dt, false);
} catch (const std::exception& e) { return fail(e.what()); }

// B sequences of S tokens: sequence b's rows start at row b S of q, k, v and out (kernels/h3sycl.cpp:1800-1815)
H3S_EXPORT int h3s_attention_batch(void* ctx, const void* q, const void* k, const void* v, int dt, int64_t B, int64_t S,
                                   int64_t H, int64_t D, int64_t stride, void* out, int out_dt) try {
    const char* fn = "h3s_attention_batch";
    if (B <= 0 || S <= 0 || H <= 0 || D <= 0) return 0;
    if (attention_checks(fn, dt, H, D, stride, out_dt, q, k, v, out)) return -1;
    Ctx* c = ctx_of(ctx, fn);
    if (!c) return -1;
    const size_t ei = (size_t) elem_size(dt), eo = (size_t) elem_size(out_dt);
    for (int64_t b = 0; b < B; ++b) {
        const size_t io = (size_t) (b * S * stride) * ei, oo = (size_t) (b * S * H * D) * eo;
        if (attention_one(c, fn, (const char*) q + io, (const char*) k + io, (const char*) v + io, dt, S, H, H, D, stride,
                          stride, (char*) out + oo, out_dt, false))
            return -1;
    }
    return 0;
} catch (const std::exception& e) { return fail(e.what()); }

// The text encoder's causal attention with grouped key/value heads (kernels/h3sycl.h:104-108, kernels/h3sycl.cpp:873-898):
// q rows of stride qs (Hq heads), k and v rows of stride kvs (Hkv heads), head h reads kv head h / (Hq / Hkv); out
// [L, Hq * D] in dt. The 16-bit form with a causal mask; any head size up to 256, as the reference.
H3S_EXPORT int h3s_attention_causal(void* ctx, const void* q, const void* k, const void* v, int dt, int64_t L, int64_t Hq,
                                    int64_t Hkv, int64_t D, int64_t qs, int64_t kvs, void* out) try {
    const char* fn = "h3s_attention_causal";
    if (L <= 0 || D <= 0) return 0;
    if (Hq <= 0 || Hkv <= 0 || Hq % Hkv != 0) return fail(std::string(fn) + ": Hq must be a multiple of Hkv");
    if (D > kAttnMaxD) return fail(std::string(fn) + ": D <= 256, Hq a multiple of Hkv (head size " + std::to_string(D) + ")");
    if (qs < Hq * D || kvs < Hkv * D) return fail(std::string(fn) + ": a row stride is shorter than a row");
    if (!dt_ok(dt)) return fail(std::string(fn) + ": unknown element type");
    if (!q || !k || !v || !out) return fail(std::string(fn) + ": q, k, v and out are required");
    Ctx* c = ctx_of(ctx, fn);
    if (!c) return -1;
    return attention_one(c, fn, q, k, v, dt, L, Hq, Hkv, D, qs, kvs, out, dt, true);
} catch (const std::exception& e) { return fail(e.what()); }
