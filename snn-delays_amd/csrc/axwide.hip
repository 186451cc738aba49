// Axonal forward scan past the sizes whose W fits one workgroup's registers (N > 256): spikes
// are scattered where they arrive, one batch row per workgroup, one neuron per lane.
//
// A spike of j enters the recurrent input at the steps of its tap run, h_j(f) W[:, j] at step
// arrival + f. Each lane keeps the KF pending sums of its own neuron in registers, so an arriving
// spike costs one row of W^T (read once, whatever the number of taps) and KF multiply-adds per
// lane; nothing is done for silent sources. Per step: the arrivals listed by the step before
// are walked in a fixed order, eight rows of W^T in flight ahead of the multiply-adds; then the
// neurons, and each wave's list of the sources arriving next. One barrier per step.
// Bound: at a few percent firing the L2 latency of the first rows and the exchange, then the rows'
// bytes (N = 512 at 3.4 %: 17 rows of 2 KB a step); past that the multiply-adds' issue, KF to an
// arrival and wave. Measured (scan, T96 B64, N 512, delays to 25; a readlane before each
// multiply-add / the row broadcast of add_pair): 3 % firing, sigma 1 249 / 198 us, sigma 3
// 341 / 242 us; 80 % firing, sigma 1 2.57 / 1.63 ms, sigma 3 4.14 / 2.19 ms. The dense product
// (axonal_fwd_kernel) takes 3.08 ms whatever the firing.
#include <algorithm>

#include "common.h"
#include "kernels.h"

namespace delrec {

namespace {
constexpr int kRows = 8;        // rows of W^T in flight (two such blocks: the lanes of a row of 16)
constexpr int kWaves = 16;
constexpr int kAhead = 4;       // steps of x loaded together

// pend[f] += h[f] of lane E of the lane's row of 16 times x0, then of lane E + 1 times x1, ..: the
// broadcast is an operand modifier of the multiply-add (the compiler makes it a move of its
// own; from a scalar register, a readlane goes before each). The s_nop covers the two wait
// states a row-modified operand needs after a vector write; the sums are written before the
// last operand is read, so they share no register with one (&).
#define DELREC_AXF(P, H, X, E) "v_fmac_f32_dpp %" P ", %" H ", %" X " row_newbcast:%" E " row_mask:0xf bank_mask:0xf\n\t"
#define DELREC_AXF2(X, E) DELREC_AXF("0", "2", X, E) DELREC_AXF("1", "3", X, E)
#define DELREC_AXF4(X, E) \
    DELREC_AXF("0", "4", X, E) DELREC_AXF("1", "5", X, E) DELREC_AXF("2", "6", X, E) DELREC_AXF("3", "7", X, E)
#define DELREC_AXF8(X, E)                                                                                         \
    DELREC_AXF("0", "8", X, E) DELREC_AXF("1", "9", X, E) DELREC_AXF("2", "10", X, E) DELREC_AXF("3", "11", X, E) \
    DELREC_AXF("4", "12", X, E) DELREC_AXF("5", "13", X, E) DELREC_AXF("6", "14", X, E) DELREC_AXF("7", "15", X, E)

template <int E>
__device__ __forceinline__ void add_pair(float x0, float x1, const float (&h)[2], float (&p)[2]) {
    asm("s_nop 1\n\t" DELREC_AXF2("4", "6") DELREC_AXF2("5", "7")
        : "+&v"(p[0]), "+&v"(p[1])
        : "v"(h[0]), "v"(h[1]), "v"(x0), "v"(x1), "n"(E), "n"(E + 1));
}
template <int E>
__device__ __forceinline__ void add_pair(float x0, float x1, const float (&h)[4], float (&p)[4]) {
    asm("s_nop 1\n\t" DELREC_AXF4("8", "10") DELREC_AXF4("9", "11")
        : "+&v"(p[0]), "+&v"(p[1]), "+&v"(p[2]), "+&v"(p[3])
        : "v"(h[0]), "v"(h[1]), "v"(h[2]), "v"(h[3]), "v"(x0), "v"(x1), "n"(E), "n"(E + 1));
}
template <int E>
__device__ __forceinline__ void add_pair(float x0, float x1, const float (&h)[8], float (&p)[8]) {
    asm("s_nop 1\n\t" DELREC_AXF8("16", "18") DELREC_AXF8("17", "19")
        : "+&v"(p[0]), "+&v"(p[1]), "+&v"(p[2]), "+&v"(p[3]), "+&v"(p[4]), "+&v"(p[5]), "+&v"(p[6]), "+&v"(p[7])
        : "v"(h[0]), "v"(h[1]), "v"(h[2]), "v"(h[3]), "v"(h[4]), "v"(h[5]), "v"(h[6]), "v"(h[7]), "v"(x0), "v"(x1),
          "n"(E), "n"(E + 1));
}
}  // namespace

// LDS: tap weights [KF][threads], arrival lists [2][16 waves][64], their lengths [2][16]
template <int KF, int HW, bool WBF>
__global__ void __launch_bounds__(1024) axonal_fwd_arrive_kernel(AxFwd p) {
    extern __shared__ float smem[];
    const int N = p.N, T = p.T, B = p.B, NT = (int)blockDim.x, nw = NT >> 6;
    const int b = blockIdx.x, i = threadIdx.x, lane = i & 63, wave = __builtin_amdgcn_readfirstlane(i >> 6);
    const bool act = i < N;
    const int ic = act ? i : 0;
    const Lif k = p.lif;
    float* htab = smem;
    uint16_t* seg = reinterpret_cast<uint16_t*>(smem + KF * NT);
    int* cnt = reinterpret_cast<int*>(seg + 2 * kWaves * 64);

    // this neuron as a source: its first lag of positive weight (>= 1) and the run's weights
    const float c = 1.0f + p.d[ic], s = p.s_uniform, s2 = s * s;
    int lo, hi;
    tap_range(c, s, p.L, lo, hi);
    if (tri_weight((float)lo, c, s, s2) <= 0.0f) lo += 1;
    lo = min(max(lo, 1), 64 * HW);
    float h[KF];
#pragma unroll
    for (int f = 0; f < KF; ++f) {
        h[f] = act && lo + f <= p.L - 1 ? tri_weight((float)(lo + f), c, s, s2) : 0.0f;
        htab[f * NT + i] = h[f];
    }
    for (int q = i; q < 2 * kWaves; q += NT) cnt[q] = 0;
    const float m = p.drop ? p.drop[(size_t)b * N + ic] : 1.0f;
    const float bias = p.bias ? p.bias[ic] : 0.0f;
    __syncthreads();

    const i32x4 rw = buffer_rsrc(p.Wt, (uint32_t)((size_t)N * N * (WBF ? 2 : 4)));
    const int wv = act ? i * (WBF ? 2 : 4) : kOutOfRange, wrow = N * (WBF ? 2 : 4);
    const size_t BN = (size_t)B * N;
    const uint32_t row_bytes = (uint32_t)BN * 4u;
    const int voff = act ? (b * N + i) * 4 : kOutOfRange;
    auto at_step = [&](const float* x, int t) {
        return step_rsrc((uint64_t)x + (uint64_t)min(t, T - 1) * row_bytes, t < T ? row_bytes : 0u);
    };
    // x of kAhead steps in registers while the next ones load
    float xq[kAhead], xn[kAhead];
#pragma unroll
    for (int q = 0; q < kAhead; ++q) xq[q] = raw_buffer_load_f32(at_step(p.x, q), voff, 0, 0);
    if (p.z) raw_buffer_store_f32(0.0f, at_step(p.z, 0), voff, 0, 0);

    float pend[KF];                                        // recurrent input of steps t .. t + KF - 1
#pragma unroll
    for (int f = 0; f < KF; ++f) pend[f] = 0.0f;
    uint64_t hist[HW];                                     // bit l - 1: the spike l steps ago
#pragma unroll
    for (int w = 0; w < HW; ++w) hist[w] = 0;
    float v = k.v0;
    uint32_t word = 0;
    const int TW = (T + 31) >> 5;

    for (int t = 0; t < T; ++t) {
        const int r = t & (kAhead - 1), sel = t & 1;
        if (r == 0) {
#pragma unroll
            for (int q = 0; q < kAhead; ++q) xn[q] = raw_buffer_load_f32(at_step(p.x, t + kAhead + q), voff, 0, 0);
        }
        // the lists' lengths, summed up to each wave's (lane w: wave w)
        const int own = lane < nw ? cnt[sel * kWaves + lane] : 0;
        int upto = own;
#pragma unroll
        for (int o = 1; o < kWaves; o <<= 1) {
            const int x = __shfl_up(upto, o);
            upto += lane >= o ? x : 0;
        }
        const int total = __builtin_amdgcn_readlane(upto, kWaves - 1);
        for (int base = 0; base < total; base += 64) {
            // lane a: arrival base + a -- its wave, its source, its weights
            const int a = base + lane;
            int w = 0, before = 0;
#pragma unroll
            for (int q = 0; q < kWaves; ++q) {
                const int e = __builtin_amdgcn_readlane(upto, q);
                w += a >= e ? 1 : 0;
                before = a >= e ? e : before;
            }
            const bool have = a < total;
            const int src = have ? seg[(sel * kWaves + w) * 64 + (a - before)] : 0;
            float hs[KF];
#pragma unroll
            for (int f = 0; f < KF; ++f) hs[f] = have ? htab[f * NT + src] : 0.0f;
            const int n = min(64, total - base);
            float wa[kRows], wb[kRows];
            auto rows = [&](int q0, float (&x)[kRows]) {
#pragma unroll
                for (int q = 0; q < kRows; ++q) {
                    const int so = __builtin_amdgcn_readlane(src, (q0 + q) & 63) * wrow;
                    x[q] = WBF ? bf16_to_f32(raw_buffer_load_u16(rw, wv, so, 0)) : raw_buffer_load_f32(rw, wv, so, 0);
                }
            };
            rows(0, wa);
            for (int q0 = 0; q0 < n; q0 += 2 * kRows) {
                float hr[KF];                              // lane E of every row of 16: arrival q0 + E's weights
#pragma unroll
                for (int f = 0; f < KF; ++f) hr[f] = __shfl(hs[f], q0 + (lane & 15));
                if (q0 + kRows < n) rows(q0 + kRows, wb);
                add_pair<0>(wa[0], wa[1], hr, pend);
                add_pair<2>(wa[2], wa[3], hr, pend);
                add_pair<4>(wa[4], wa[5], hr, pend);
                add_pair<6>(wa[6], wa[7], hr, pend);
                if (q0 + kRows < n) {
                    if (q0 + 2 * kRows < n) rows(q0 + 2 * kRows, wa);
                    add_pair<8>(wb[0], wb[1], hr, pend);
                    add_pair<10>(wb[2], wb[3], hr, pend);
                    add_pair<12>(wb[4], wb[5], hr, pend);
                    add_pair<14>(wb[6], wb[7], hr, pend);
                }
            }
        }
        float xv = xq[0];
#pragma unroll
        for (int q = 1; q < kAhead; ++q) xv = r == q ? xq[q] : xv;
        const float rec = pend[0] + bias;
        const float u = lif_charge(k, v, xv + rec * m);
        const float y = lif_fire(k, u);
        v = lif_reset(k, u, y);
#pragma unroll
        for (int f = 0; f < KF; ++f) pend[f] = f + 1 < KF ? pend[f + 1] : 0.0f;
        const uint32_t yb = y != 0.0f && act ? 1u : 0u;
#pragma unroll
        for (int w = HW - 1; w > 0; --w) hist[w] = (hist[w] << 1) | (hist[w - 1] >> 63);
        hist[0] = (hist[0] << 1) | (uint64_t)yb;
        word |= yb << (t & 31);
        // the run's spikes at step t + 1: bit f of `run` = y(t + 1 - lo - f)
        uint64_t run = hist[0];
        if constexpr (HW > 1) {
            const int kb = (lo - 1) >> 6;
            run = 0;
            uint64_t over = 0;
#pragma unroll
            for (int w = 0; w < HW; ++w) {
                run = kb == w ? hist[w] : run;
                over = kb + 1 == w ? hist[w] : over;
            }
            const int sh = (lo - 1) & 63;
            run = sh ? (run >> sh) | (over << (64 - sh)) : run;
        } else {
            run >>= lo - 1;
        }
        const bool next = (run & 1ull) != 0;               // arrives at t + 1
        const uint64_t bal = __ballot(next);
        if (next) seg[((sel ^ 1) * kWaves + wave) * 64 + __popcll(bal & ((1ull << lane) - 1ull))] = (uint16_t)i;
        if (lane == 0) cnt[(sel ^ 1) * kWaves + wave] = __popcll(bal);
        raw_buffer_store_f32(y, at_step(p.y, t), voff, 0, 0);
        raw_buffer_store_f32(u, at_step(p.u, t), voff, 0, 0);
        if (p.rec) raw_buffer_store_f32(rec, at_step(p.rec, t), voff, 0, 0);
        if (p.z) {
            float z = 0.0f;
#pragma unroll
            for (int f = 0; f < KF; ++f) z += h[f] * (float)((run >> f) & 1ull);
            raw_buffer_store_f32(z, at_step(p.z, t + 1), voff, 0, 0);
        }
        if ((t & 31) == 31 || t == T - 1) {
            if (act) p.bits[((size_t)b * TW + (t >> 5)) * N + i] = word;
            word = 0;
        }
        if (r == kAhead - 1) {
#pragma unroll
            for (int q = 0; q < kAhead; ++q) xq[q] = xn[q];
        }
        barrier_lds();
    }
}

template <int KF, int HW>
static void launch_arrive(const AxFwd& p, int block, size_t lds, hipStream_t s) {
    if (p.w_bf16) {
        ensure_lds((const void*)axonal_fwd_arrive_kernel<KF, HW, true>, lds);
        hipLaunchKernelGGL((axonal_fwd_arrive_kernel<KF, HW, true>), dim3(p.B), dim3(block), lds, s, p);
    } else {
        ensure_lds((const void*)axonal_fwd_arrive_kernel<KF, HW, false>, lds);
        hipLaunchKernelGGL((axonal_fwd_arrive_kernel<KF, HW, false>), dim3(p.B), dim3(block), lds, s, p);
    }
}

bool launch_axonal_fwd_arrive(const AxFwd& p, int kf, int hw, hipStream_t s) {
    const int block = (p.N + 63) / 64 * 64;
    const size_t lds = (size_t)kf * block * sizeof(float) + 2 * kWaves * 64 * sizeof(uint16_t) + 2 * kWaves * sizeof(int);
#define DELREC_AXW(KFV, HWV) if (kf == KFV && hw == HWV) { launch_arrive<KFV, HWV>(p, block, lds, s); return true; }
    DELREC_AXW(2, 1) DELREC_AXW(2, 2) DELREC_AXW(2, 4)
    DELREC_AXW(4, 1) DELREC_AXW(4, 2) DELREC_AXW(4, 4)
    DELREC_AXW(8, 1) DELREC_AXW(8, 2) DELREC_AXW(8, 4)
#undef DELREC_AXW
    return false;
}

}  // namespace delrec
