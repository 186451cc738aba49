// Reverse-time scan of a layer with a delay of its own for each connection and one half-width s,
// fp32, one batch row per workgroup.
//
// The triangle's weights are linear in the delay's fraction f between knots. With n = floor(d),
// m = floor(s), r = s - m and the lags n + 1 + q,
//   s^2 gfut = A(n) + f D(n) + max(0, r - f) g(n + 1 - m) + max(0, f - (1 - r)) g(n + 2 + m),
//   A(n) = sum_{q <= 0} (s + q) g(n + 1 + q) + sum_{q >= 1} (s - q) g(n + 1 + q),
//   D(n) = sum_{q >= 1} g(n + 1 + q) - sum_{q <= 0} g(n + 1 + q),   -m < q <= m,
// g(l) = gr(t + l), 0 where l < 1. A and D are one receiver's, the same for all its connections:
// its thread adds each new gr to the 2 m slots (time t + n, mod R) of its LDS row that contain it,
// and a connection reads one pair and takes two multiply-adds, whatever the number of taps
// (and, where s is no whole number, two more values and multiply-adds). Slots hold only what
// is known, so lags below 1 drop out by themselves.
// A connection is 8 bytes: W in fp32 and (n mod R as a byte offset) << 24 | f in 23 bits, read as
// the float 1 + f (the pair holds A - D). Lanes are sources, a wave reads one receiver row at a
// time: distinct slots are distinct banks, equal ones broadcast.
// Bound: LDS, 85 % of the kernel's clocks at T250 B256 N256 sigma 1, two thirds of that conflicts (the
// pairs of a wave's lanes, and the neurons' own rows, which all start in one bank); then the
// operands from L2 (524 KB a step, 36 of 64 B/clk per CU) and vector issue (43 %). Where s is no whole
// number the kernel spills 23 registers of 128.
// Measured (scan), with the taps walked one by one (syn_bwd_kernel) / with the tables:
//   T250 B256 N256 sigma 1 8.51 / 1.64 ms (34 / 6.6 us a step); T48 B64: N 100 sigma 1 0.74 / 0.11,
//   N 160 sigma 0.4 0.73 / 0.29, N 256 sigma 3 2.16 / 0.38, N 512 sigma 0 2.47 / 0.84 ms.
#include <algorithm>

#include "common.h"
#include "kernels.h"

namespace delrec {

__global__ void __launch_bounds__(256) syn_lin_pack_kernel(SynLin p, uint4* wq, uint4* fq, const void* W,
                                                           const float* d) {
    const int total = p.NC * p.Ns;
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= total) return;
    const int c = q / p.Ns, j = q - c * p.Ns, N = p.N, m = p.m;
    const int unit = p.R == 32 ? 8 : 4;
    uint32_t w[16], f[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int i = c * 16 + e;
        const bool ok = i < N && j < N;
        const size_t at = ok ? (size_t)i * N + j : 0;
        float wv = ok ? load_w(W, p.w_bf16, at) : 0.0f;
        const float dv = ok ? d[at] : 0.0f;
        float fl = floorf(dv);
        uint32_t fr = (uint32_t)rintf((dv - fl) * 8388608.0f);
        int n = (int)fl;
        if (fr >= 8388608u) {                              // rounded up to the next step
            fr = 0;
            n += 1;
        }
        if (n < -m - 1 || dv != dv) {                      // no lag of positive weight: times 0
            n = 0;
            fr = 0;
            wv *= 0.0f;
        }
        if (n > p.L) {                                     // no such delay in the stated window
            n = 0;
            wv = __builtin_nanf("");
        }
        w[e] = __float_as_uint(wv);
        f[e] = ((uint32_t)((n * unit) & 0xFF) << 24) | fr;
    }
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        wq[(size_t)(c * 4 + h) * p.Ns + j] = make_uint4(w[4 * h], w[4 * h + 1], w[4 * h + 2], w[4 * h + 3]);
        fq[(size_t)(c * 4 + h) * p.Ns + j] = make_uint4(f[4 * h], f[4 * h + 1], f[4 * h + 2], f[4 * h + 3]);
    }
}

// R slots: 32 (a row: 32 pairs) or 64 (a row: 64 A, 64 D); FRAC: s is no whole number (a row ends
// with the R values of gr). LDS: rows, then partial sums [slices][Ns].
template <int R, bool FRAC>
__global__ void __launch_bounds__(1024) syn_lin_bwd_kernel(SynLin p) {
    extern __shared__ float smem[];
    constexpr int ROW = R * (FRAC ? 3 : 2);                // words per receiver
    constexpr int PF = 2;                                  // steps of gy / u loaded together
    const int N = p.N, T = p.T, B = p.B, Ns = p.Ns, NC = p.NC, m = p.m;
    const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nsb = Ns >> 6, slice = wave / nsb, sb = wave % nsb;   // slice of the receivers, block of sources
    const int c0 = min(slice * p.per, NC), c1 = min(c0 + p.per, NC);
    const float sv = p.s_uniform, r1 = 1.0f + (sv - (float)m), r2 = 2.0f - (sv - (float)m);
    float* const red = smem + (size_t)NC * 16 * ROW;
    for (int q = tid; q < NC * 16 * ROW + p.slices * Ns; q += blockDim.x) smem[q] = 0.0f;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float*)smem;

    const i32x4 rw = buffer_rsrc(p.wq, (uint32_t)((size_t)NC * 4 * Ns * 16));
    const i32x4 rf = buffer_rsrc(p.fq, (uint32_t)((size_t)NC * 4 * Ns * 16));
    const int vo = (sb * 64 + lane) * 16;
    struct Chunk { uint4 w[4], f[4]; };
    auto load4 = [](i32x4 rs, int voff, int soff) {
        const i32x4 v = raw_buffer_load_i32x4(rs, voff, soff, 0);
        return make_uint4((uint32_t)v.x, (uint32_t)v.y, (uint32_t)v.z, (uint32_t)v.w);
    };
    auto fetch = [&](Chunk& ch, int h, int c) {
        ch.w[h] = load4(rw, vo, (c * 4 + h) * Ns * 16);
        ch.f[h] = load4(rf, vo, (c * 4 + h) * Ns * 16);
    };
    // acc += the chunk's 16 connections at step byte st (t as a slot byte << 24); then the operands
    // of chunk nc come in
    auto sum_chunk = [&](Chunk& ch, int c, uint32_t st, int nc, float acc) {
        const uint32_t cb = lds0 + (uint32_t)c * (16 * ROW * 4);
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            const uint32_t fw[4] = {ch.f[h].x, ch.f[h].y, ch.f[h].z, ch.f[h].w};
            const uint32_t ww[4] = {ch.w[h].x, ch.w[h].y, ch.w[h].z, ch.w[h].w};
            float A[4], D[4], g1[4], g2[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (FRAC && q == 2) __builtin_amdgcn_sched_barrier(0);
                const uint32_t sl = (fw[q] + st) >> 24;    // the slot's byte offset, wrapped by the byte
                const auto* x = (const __attribute__((address_space(3))) float*)(uintptr_t)(cb + sl) + (4 * h + q) * ROW;
                A[q] = x[0];
                D[q] = x[R == 32 ? 1 : R];
                if constexpr (FRAC) {
                    const uint32_t so = R == 32 ? sl >> 1 : sl;         // (4 bytes a slot here)
                    const auto* y = (const __attribute__((address_space(3))) float*)(uintptr_t)(cb + 2 * R * 4) + (4 * h + q) * ROW;
                    g1[q] = y[((so >> 2) + (uint32_t)(R + 1 - m)) & (R - 1)];
                    g2[q] = y[((so >> 2) + (uint32_t)(2 + m)) & (R - 1)];
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float f1 = __uint_as_float((fw[q] & 0x7FFFFFu) | 0x3F800000u);   // 1 + f
                float v = fmaf(f1, D[q], A[q]);
                if constexpr (FRAC) {
                    v = fmaf(fmaxf(r1 - f1, 0.0f), g1[q], v);
                    v = fmaf(fmaxf(f1 - r2, 0.0f), g2[q], v);
                }
                acc = fmaf(__uint_as_float(ww[q]), v, acc);
            }
            fetch(ch, h, nc);
            __builtin_amdgcn_sched_barrier(0);             // bounds the reads in flight (registers)
        }
        return acc;
    };
    Chunk ch;
#pragma unroll
    for (int h = 0; h < 4; ++h) fetch(ch, h, min(c0, NC - 1));

    // thread j: neuron j
    const bool act = tid < N;
    const int j = act ? tid : 0;
    const Lif k = p.lif;
    const float mk = p.drop ? p.drop[(size_t)b * N + j] : 1.0f;
    const float is2 = 1.0f / (sv * sv);
    float* const own = smem + (size_t)j * ROW;
    const size_t BN = (size_t)B * N;
    const uint32_t row_bytes = (uint32_t)BN * 4u;
    const int voff = act ? (b * N + j) * 4 : kOutOfRange;
    auto at_step = [&](const float* x, int t) {
        return step_rsrc((uint64_t)x + (uint64_t)max(t, 0) * row_bytes, t >= 0 ? row_bytes : 0u);
    };
    float gq[PF], uq[PF], gn[PF], un[PF];
    auto load_steps = [&](int t, float (&g)[PF], float (&u)[PF]) {
#pragma unroll
        for (int q = 0; q < PF; ++q) {
            g[q] = raw_buffer_load_f32(at_step(p.gy, t - q), voff, 0, 0);
            u[q] = raw_buffer_load_f32(at_step(p.u, t - q), voff, 0, 0);
        }
    };
    const bool neurons = wave * 64 < N;
    if (neurons) load_steps(T - 1, gq, uq);
    float lam = 0.0f, dbacc = 0.0f;
    __syncthreads();

    for (int t = T - 1; t >= 0; --t) {
        const int r = (T - 1 - t) & (PF - 1);
        if (neurons && r == 0) load_steps(t - PF, gn, un);
        const uint32_t st = (uint32_t)((t * (R == 32 ? 8 : 4)) & 0xFF) << 24;
        float acc = 0.0f;
#pragma unroll 1
        for (int c = c0; c < c1; ++c) acc = sum_chunk(ch, c, st, c + 1 < c1 ? c + 1 : c0, acc);
        red[slice * Ns + sb * 64 + lane] = acc;
        barrier_lds();
        if (neurons) {
            float gf = 0.0f;
#pragma unroll 4
            for (int q = 0; q < p.slices; ++q) gf += red[q * Ns + j];
            gf *= is2;
            const float u = r == 0 ? uq[0] : uq[1], gyv = r == 0 ? gq[0] : gq[1];
            const float y = lif_fire(k, u);
            const float du = lif_backward(k, gyv + gf, u, y, lam);
            lam = k.decay * du;
            const float da = lif_dx(k, du);
            const float gr = da * mk;
            if (act) {
                // gr(t) is lag n + 1 + q of the slots of time t - 1 - q; the slot of q = m is new, the
                // one before it cleared
                auto pair = [&](int time) { return own + (R == 32 ? 2 : 1) * (time & (R - 1)); };
                constexpr int DO = R == 32 ? 1 : R;
#pragma unroll 2
                for (int q = 1 - m; q < m; ++q) {
                    float* x = pair(t - 1 - q);
                    const float c1q = q >= 1 ? 1.0f : -1.0f, c0q = (q >= 1 ? sv - (float)q : sv + (float)q) - c1q;
                    const float a = x[0], dd = x[DO];
                    x[0] = fmaf(c0q, gr, a);
                    x[DO] = fmaf(c1q, gr, dd);
                }
                float* x = pair(t - 1 - m);
                x[0] = (sv - (float)m - 1.0f) * gr;        // q = m
                x[DO] = gr;
                x = pair(t - 2 - m);
                x[0] = 0.0f;
                x[DO] = 0.0f;
                if constexpr (FRAC) {
                    own[2 * R + (t & (R - 1))] = gr;
                    own[2 * R + ((t - 2 * m - 2) & (R - 1))] = 0.0f;    // times up to t - 1 read as 0
                }
            }
            raw_buffer_store_f32(da, at_step(p.dx, t), voff, 0, 0);
            if (p.gr) raw_buffer_store_f32(gr, at_step(p.gr, t), voff, 0, 0);
            dbacc += gr;
            if (r == PF - 1) {
#pragma unroll
                for (int q = 0; q < PF; ++q) {
                    gq[q] = gn[q];
                    uq[q] = un[q];
                }
            }
        }
        barrier_lds();
    }
    if (act) p.part[(size_t)b * N + j] = dbacc;
}

SynLinShape syn_lin_shape(int N, int L, float s, size_t max_lds) {
    SynLinShape q{};
    if (N < 1 || N > 1024 || !(s >= 1.0f) || s > 16.0f || L < 2) return q;
    q.m = (int)floorf(s);
    q.frac = s > (float)q.m;
    // slots at once: the longest delay (n <= L - 2 - m, one more where its fraction rounds up), the
    // 2 m slots a step adds to, the cleared one; gr's own ring reaches m + 2 further either way
    const int slots = L + 3 + (q.frac ? 2 * q.m + 4 : 0);
    q.R = slots <= 32 ? 32 : slots <= 64 ? 64 : 0;
    if (!q.R) return q;
    q.NC = (N + 15) / 16;
    const int nsb = (N + 63) / 64;
    q.Ns = nsb * 64;
    q.slices = std::max(1, std::min(16 / nsb, q.NC));
    q.per = (q.NC + q.slices - 1) / q.slices;
    q.block = nsb * q.slices * 64;
    q.lds = ((size_t)q.NC * 16 * q.R * (q.frac ? 3 : 2) + (size_t)q.slices * q.Ns) * sizeof(float);
    q.pack = (size_t)q.NC * 4 * q.Ns;
    q.ok = q.lds <= max_lds;
    return q;
}

bool launch_syn_lin_bwd(const SynLin& p, const SynLinShape& q, uint4* wq, uint4* fq, const void* W, const float* d,
                        hipStream_t s) {
    hipLaunchKernelGGL(syn_lin_pack_kernel, dim3((q.NC * q.Ns + 255) / 256), dim3(256), 0, s, p, wq, fq, W, d);
#define DELREC_SYNLIN(RV, FV)                                                                     \
    if (q.R == RV && q.frac == FV) {                                                              \
        ensure_lds((const void*)syn_lin_bwd_kernel<RV, FV>, q.lds);                               \
        hipLaunchKernelGGL((syn_lin_bwd_kernel<RV, FV>), dim3(p.B), dim3(q.block), q.lds, s, p);  \
        return true;                                                                              \
    }
    DELREC_SYNLIN(32, false) DELREC_SYNLIN(32, true) DELREC_SYNLIN(64, false) DELREC_SYNLIN(64, true)
#undef DELREC_SYNLIN
    return false;
}

}  // namespace delrec
