// steps.hip - what a sampler step fixes for every block, on the device (engine/h3-core/src/dit.rs:155-203, a host
// loop in the reference): h3s_adaln_tables (the six AdaLN tables of a block from the timestep embeddings) and
// h3s_rotations (the (cos, sin) table of every token's position).
#include <cmath>

#include "common.h"

namespace h3 {

// out[ci][(r m + mi) C + i] = b[o] + sum_k fl(w[o, k] t[r, k]), o = mi 6 C + ci C + i: the sum in k order from -0.0 in
// float32 (dit.rs:163-170, Rust's f32 Sum), one multiply and one add a term (no fused multiply-add). Bound by the read of w.
// A wavefront takes 64 consecutive o and NR timestep rows at once (w is read once for them; blockIdx.y counts the groups of
// NR rows, the last one's missing rows repeating the last row, not stored); a tile of 64 o x 32 k goes through registers to
// LDS in 16-byte pieces that cover whole 128-byte lines, two tiles in flight while the one before is summed, and each lane
// runs its own o's NR sums (t[r, k] is a scalar operand). The LDS rows are 36 floats apart, so 16 lanes' 16-byte reads touch
// every bank once. VEC = 1 (rows that are not whole 16-byte pieces) loads single floats the same way. 96768 x 256 floats with
// 2 timesteps, and the rotations of 2159 tokens: 185.6 -> 22.6 us (the tables alone 153 -> 20.5: 64 dependent row loads a
// tile and w read once a timestep; the 101 MB take 20 us at the rate of a large copy). All groups in one launch: with few
// outputs and many timesteps a launch a group leaves the device idle (R = 1000, 384 x 256 floats: 3251 us, 99 with one launch
// of a row a block, 17.6 here).
constexpr int kTabK = 32, kTabStride = kTabK + 4;
template <int NR, int VEC>
__global__ __launch_bounds__(64) void adaln_tables_kernel(const float* __restrict__ w, const float* __restrict__ b,
                                                          const float* __restrict__ t, int64_t R, int64_t td, int64_t m,
                                                          int64_t C, float* __restrict__ out) {
    constexpr int LPR = kTabK / VEC, RPL = 64 / LPR, NL = 64 / RPL;   // lanes a row, rows a load, loads a tile
    typedef float fvec __attribute__((ext_vector_type(VEC)));
    __shared__ __attribute__((aligned(16))) float tile[64 * kTabStride];
    const int64_t r0 = (int64_t) blockIdx.y * NR;
    int64_t row[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) row[r] = r0 + r < R ? r0 + r : R - 1;
    const int lane = threadIdx.x, lr = lane / LPR, lk = lane % LPR * VEC;
    const int64_t nout = 6 * m * C, o0 = (int64_t) blockIdx.x * 64, o = o0 + lane;
    float sum[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) sum[r] = -0.0f;
    // rows past the last o read the last one, and a tile's columns past td are not read (and not summed)
    fvec buf[2][NL];
    auto fetch = [&](fvec (&f)[NL], int64_t k0) {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int64_t row = o0 + i * RPL + lr;
            const float* p = w + (row < nout ? row : nout - 1) * td + k0 + lk;
            f[i] = fvec(0.0f);
            if (k0 + lk < td) f[i] = *reinterpret_cast<const fvec*>(p);
        }
    };
    auto step = [&](fvec (&f)[NL], int64_t k0) {
#pragma unroll
        for (int i = 0; i < NL; ++i) *reinterpret_cast<fvec*>(&tile[(i * RPL + lr) * kTabStride + lk]) = f[i];
        fetch(f, k0 + 2 * kTabK);
        lds_barrier();
        const float* mine = &tile[lane * kTabStride];
        const float* tk = t + k0;
        if (k0 + kTabK <= td) {
#pragma unroll
            for (int k = 0; k < kTabK; k += 4) {
                const float4 v = *reinterpret_cast<const float4*>(mine + k);
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    const float* tr = tk + row[r] * td + k;
                    sum[r] = sum[r] + v.x * tr[0];
                    sum[r] = sum[r] + v.y * tr[1];
                    sum[r] = sum[r] + v.z * tr[2];
                    sum[r] = sum[r] + v.w * tr[3];
                }
            }
        } else {
            for (int k = 0; k < td - k0; ++k) {
                const float v = mine[k];
#pragma unroll
                for (int r = 0; r < NR; ++r) sum[r] = sum[r] + v * tk[row[r] * td + k];
            }
        }
        lds_barrier();
    };
    fetch(buf[0], 0);
    fetch(buf[1], kTabK);
    for (int64_t k0 = 0; k0 < td; k0 += 2 * kTabK) {
        step(buf[0], k0);
        if (k0 + kTabK < td) step(buf[1], k0 + kTabK);
    }
    if (o >= nout) return;
    const int64_t mi = o / (6 * C), ci = (o / C) % 6, i = o % C;
    float* p = out + ci * R * m * C + mi * C + i;
    const float bo = b[o];
#pragma unroll
    for (int r = 0; r < NR; ++r)
        if (r0 + r < R) p[(r0 + r) * m * C] = bo + sum[r];
}

template <int VEC>
static void adaln_tables(Ctx* c, const float* w, const float* b, const float* t, int64_t R, int64_t td, int64_t m, int64_t C,
                         float* out) {
    const int64_t nr = R < 4 ? R : 4;
    const dim3 grid((unsigned) ((6 * m * C + 63) / 64), (unsigned) ((R + nr - 1) / nr));
    if (nr == 4) adaln_tables_kernel<4, VEC><<<grid, 64, 0, c->stream>>>(w, b, t, R, td, m, C, out);
    else if (nr == 3) adaln_tables_kernel<3, VEC><<<grid, 64, 0, c->stream>>>(w, b, t, R, td, m, C, out);
    else if (nr == 2) adaln_tables_kernel<2, VEC><<<grid, 64, 0, c->stream>>>(w, b, t, R, td, m, C, out);
    else adaln_tables_kernel<1, VEC><<<grid, 64, 0, c->stream>>>(w, b, t, R, td, m, C, out);
}

// cs[s][a n + f] = (cos x, sin x), x = fl((float) pos[s, a] * inv_freq[f]) (dit.rs:190-203); cos and sin of the float
// argument evaluated in float64 and rounded once, so they are the correctly rounded float32 values. One sincos (one
// argument reduction) and one 8-byte store a pair.
__global__ __launch_bounds__(256) void rotations_kernel(const double* __restrict__ pos, int64_t S, const float* __restrict__ inv,
                                                        int64_t n, float* __restrict__ cs) {
    const int64_t id = (int64_t) blockIdx.x * 256 + threadIdx.x, total = S * 3 * n;
    if (id >= total) return;
    const int64_t f = id % n, sa = id / n;                  // sa = s * 3 + a
    const float x = (float) pos[sa] * inv[f];
    double si, co;
    sincos((double) x, &si, &co);
    cs[2 * id] = (float) co;
    cs[2 * id + 1] = (float) si;
}

}  // namespace h3

using namespace h3;

H3S_EXPORT int h3s_adaln_tables(void* ctx, const float* w, const float* b, const float* t_emb, int64_t R, int64_t t_dim,
                                int64_t m, int64_t C, float* out) try {
    const char* fn = "h3s_adaln_tables";
    if (R <= 0 || t_dim <= 0 || m <= 0 || C <= 0) return 0;
    if (!w || !b || !t_emb || !out) return fail(std::string(fn) + ": w, b, t_emb and out are required");
    // (a bound of the interface, since a timestep row was a block of the grid's second dimension)
    if (R > 65535) return fail(std::string(fn) + ": at most 65535 timestep rows");
    Ctx* c = ctx_of(ctx, fn);
    if (!c) return -1;
    if (t_dim % 4 == 0 && aligned16(w)) adaln_tables<4>(c, w, b, t_emb, R, t_dim, m, C, out);
    else adaln_tables<1>(c, w, b, t_emb, R, t_dim, m, C, out);
    return launched(fn);
} catch (const std::exception& e) { return fail(e.what()); }

H3S_EXPORT int h3s_rotations(void* ctx, const double* positions, int64_t S, const float* inv_freq, int64_t n, float* cs) try {
    const char* fn = "h3s_rotations";
    if (S <= 0 || n <= 0) return 0;
    if (!positions || !inv_freq || !cs) return fail(std::string(fn) + ": positions, inv_freq and cs are required");
    Ctx* c = ctx_of(ctx, fn);
    if (!c) return -1;
    const int64_t total = S * 3 * n;
    rotations_kernel<<<(unsigned) ((total + 255) / 256), 256, 0, c->stream>>>(positions, S, inv_freq, n, cs);
    return launched(fn);
} catch (const std::exception& e) { return fail(e.what()); }
