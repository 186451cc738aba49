// Reverse-time scan of a layer whose delays differ between a source's receivers by whole
// steps only (hybrid: base_j + integer offset_ij; axonal: no offset), fp32 arithmetic, one
// batch row per workgroup.
//
// With e_ij = off_ij - min off and lo_j the first lag of positive weight at the smallest offset,
//   gfut_j(t) = sum_f h_j(f) G_j(t + lo_j + f),   G_j(tau) = sum_i W[i,j] gr_i(tau + e_ij):
// one multiply-add per connection and step. G_j(tau) is needed at step tau - lo_j and its
// terms are known from step tau - 1 on, so a source may form P of its G together: the weight,
// its offset byte and the LDS address are then fetched and decoded once for P multiply-adds
// (the P values of gr are consecutive slots of the receiver's ring row), and with lo_j >= 2 P
// the work of a block is spread evenly over P steps, a P-th of the receivers in each, and none
// of it waits for the step's own gr. Sources are taken in first-lag order, sixteen to a group:
//   far groups (smallest first lag 4 .. 7: blocks of 2 steps, 8 or more: of 4) belong to one
//     wave each, dealt out in alternating order; their sums run beside the step's neurons;
//   near groups (lo = 1 .. 3) form G(t + 1) in step t: their receivers are split over all the
//     waves, whose partial sums meet in LDS before the step's neurons;
//   sources that start at lags <= 0 (half-widths over 1 near the delay 0) also need G(t),
//     G(t - 1), .. over the connections whose lag is still >= 1 -- the slots of the steps not
//     yet formed hold 0, so these are the same run of slots, started earlier.
//
// Bound: the multiply-adds' issue (with offsets: one, an address and a share of the decode for each
// connection of a block), then the LDS reads of gr (4 bytes per connection and step at 128 B/clk)
// and the two exchanges of a step. Share of the kernel's clocks, from counters:
//   T256 B256 N512 sigma 0, 9 offsets, bf16 W: vector issue 83 %, LDS 58 % (1 % of it conflicts)
//   T250 B128 N256 sigma 1, 5 offsets, fp32 W: vector issue 68 %, LDS 47 % (4 % conflicts)
//   axonal T250 B256 N512 sigma 1, fp32 W: vector issue 64 %, LDS 20 % (one read serves 16
//     receivers' multiply-adds), operands from L2 30 B/clk a CU
// Measured (scan): those three 1.7 ms (2.2 ms with syn_bwd_hyb_g), 0.65 ms, 2.6 us a step (23.5 ms
// with the gather per tap, syn_bwd_kernel) and 1.56 ms (8.70 ms with the dense product streamed per
// step, axonal_bwd_kernel). A group's whole block taken in one step by its own wave alone: 5.2
// ms at N = 512 (one wave per SIMD at a time hides nothing); neurons on the summing waves instead
// of waves of their own: 2.0 ms. Registers (of 128): runs of 1 and 2 slots spill up to 8; of 4 37
// to 46, and of 8 137 to 154, with four neurons a lane; scalar ones spill to lanes of vector
// registers (48 to 80 bytes of scratch a lane).
#include <algorithm>

#include "common.h"
#include "kernels.h"

namespace delrec {

namespace {

constexpr int kTapsMax = 12;

// First lag of positive weight of a triangle of half-width s around c = 1 + d.
__device__ __forceinline__ int first_lag(float c, float s) {
    int lo = (int)ceilf(c - s);
    if (fabsf((float)(lo - 1) - c) <= s) lo -= 1;
    if (fabsf((float)lo - c) > s) lo += 1;
    if (s - fabsf((float)lo - c) <= 0.0f) lo += 1;
    return lo;
}

// acc[n] += sum over q < 4 of w[q] * (g[n] of lane E + q of the lane's row of 16): the broadcast is
// an operand modifier of the multiply-add (the compiler makes it a move of its own). The s_nop
// covers the two wait states a row-modified operand needs after a vector write; the sums are
// written before the last operand is read, so they share no register with one (&).
template <int E>
__device__ __forceinline__ void add_rows(const float (&w)[4], const float (&g)[1], float (&acc)[1]) {
    asm("s_nop 1\n\t"
        "v_fmac_f32_dpp %0, %1, %2 row_newbcast:%6 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %3 row_newbcast:%7 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %4 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %1, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf"
        : "+&v"(acc[0])
        : "v"(g[0]), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "n"(E), "n"(E + 1), "n"(E + 2), "n"(E + 3));
}

#define DELREC_FMAC2(W, E)                                                      \
    "v_fmac_f32_dpp %0, %2, " W " row_newbcast:" E " row_mask:0xf bank_mask:0xf\n\t" \
    "v_fmac_f32_dpp %1, %3, " W " row_newbcast:" E " row_mask:0xf bank_mask:0xf\n\t"
template <int E>
__device__ __forceinline__ void add_rows(const float (&w)[4], const float (&g)[2], float (&acc)[2]) {
    asm("s_nop 1\n\t" DELREC_FMAC2("%4", "%8") DELREC_FMAC2("%5", "%9") DELREC_FMAC2("%6", "%10") DELREC_FMAC2("%7", "%11")
        : "+&v"(acc[0]), "+&v"(acc[1])
        : "v"(g[0]), "v"(g[1]), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "n"(E), "n"(E + 1), "n"(E + 2), "n"(E + 3));
}

#define DELREC_FMAC4(W, E)                                                      \
    "v_fmac_f32_dpp %0, %4, " W " row_newbcast:" E " row_mask:0xf bank_mask:0xf\n\t" \
    "v_fmac_f32_dpp %1, %5, " W " row_newbcast:" E " row_mask:0xf bank_mask:0xf\n\t" \
    "v_fmac_f32_dpp %2, %6, " W " row_newbcast:" E " row_mask:0xf bank_mask:0xf\n\t" \
    "v_fmac_f32_dpp %3, %7, " W " row_newbcast:" E " row_mask:0xf bank_mask:0xf\n\t"
template <int E>
__device__ __forceinline__ void add_rows(const float (&w)[4], const float (&g)[4], float (&acc)[4]) {
    asm("s_nop 1\n\t" DELREC_FMAC4("%8", "%12") DELREC_FMAC4("%9", "%13") DELREC_FMAC4("%10", "%14") DELREC_FMAC4("%11", "%15")
        : "+&v"(acc[0]), "+&v"(acc[1]), "+&v"(acc[2]), "+&v"(acc[3])
        : "v"(g[0]), "v"(g[1]), "v"(g[2]), "v"(g[3]), "v"(w[0]), "v"(w[1]), "v"(w[2]), "v"(w[3]), "n"(E), "n"(E + 1),
          "n"(E + 2), "n"(E + 3));
}

}  // namespace

// order[k] = the source with the k-th smallest (first lag, index), rank its inverse. One workgroup, N <= 1024:
// each thread ranks one source against all keys, four per LDS read. *wrong: the device data
// contradict what the caller stated -- the offsets span more than D steps, or a source starts
// before the lag that early runs of NT slots reach.
__global__ void __launch_bounds__(1024) hyb_block_order_kernel(const float* base, float sv, int N, const int* meta,
                                                               int NT, int D, int* order, int* rank, int* wrong) {
    __shared__ __align__(16) int key[1024];
    const int j = threadIdx.x;
    const int kj = j < N ? first_lag(1.0f + base[j], sv) : 0x7fffffff;
    key[j] = kj;
    const bool early = __syncthreads_or(meta && j < N && kj + meta[1] < 2 - NT) != 0;
    if (j == 0) *wrong = meta && (early || meta[2] - meta[1] + 1 > D) ? 1 : 0;
    if (j >= N) return;
    int pos = 0;
    for (int q = 0; q < N; q += 4) {
        const int4 v = *reinterpret_cast<const int4*>(key + q);
        pos += (v.x < kj || (v.x == kj && q < j)) + (v.y < kj || (v.y == kj && q + 1 < j)) +
               (v.z < kj || (v.z == kj && q + 2 < j)) + (v.w < kj || (v.w == kj && q + 3 < j));
    }
    order[pos] = j;
    rank[j] = pos;
}

// The scan's operands in lane order: chunk c of 16 receivers, lane slot js = source order[js],
//   wq[(c * WV + h) * Ns + js]: the weights of receivers 16 c + 4 h .. (bf16: 8 h ..), WV uint4,
//   oq[c * Ns + js]: 16 bytes 4 (off - min off);
// zero past N in either direction. Where the general scan runs in its place: that one's blocked
// copies (SynBwd::Wt, offt).
template <bool WBF>
__global__ void __launch_bounds__(256) hyb_block_pack_kernel(HybBlk p, uint4* wq, uint4* oq, const void* W,
                                                             const int8_t* off) {
    constexpr int WV = WBF ? 2 : 4;
    const int N = p.N, total = 4 * p.NCl * p.Ns;
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= total) return;
    const int c = q / p.Ns, js = q - c * p.Ns;
    if (p.wt && *p.wrong) {
        if (c * 16 >= N || js >= N) return;
        for (int e = 0; e < 16; ++e) {
            const int i = c * 16 + e;
            const size_t to = ((size_t)c * N + js) * 16 + e, at = (size_t)i * N + js;
            if constexpr (WBF) static_cast<uint16_t*>(p.wt)[to] = i < N ? static_cast<const uint16_t*>(W)[at] : 0;
            else static_cast<uint32_t*>(p.wt)[to] = i < N ? static_cast<const uint32_t*>(W)[at] : 0u;
            p.offt[to] = i < N ? off[at] : 0;
        }
        return;
    }
    const int j = js < N ? p.order[js] : 0;
    const int omin = off ? p.meta[1] : 0;
    uint32_t w[WV * 4], o[4] = {0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < WV * 4; ++e) w[e] = 0;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int i = c * 16 + e;
        const bool ok = i < N && js < N;
        const size_t at = ok ? (size_t)i * N + j : 0;
        if constexpr (WBF) {
            const uint32_t v = ok ? static_cast<const uint16_t*>(W)[at] : 0u;
            w[e >> 1] |= v << (16 * (e & 1));
        } else {
            w[e] = ok ? static_cast<const uint32_t*>(W)[at] : 0u;
        }
        if (off && ok) o[e >> 2] |= (uint32_t)(((off[at] - omin) * 4) & 0xFF) << (8 * (e & 3));
    }
#pragma unroll
    for (int h = 0; h < WV; ++h)
        wq[(size_t)(c * WV + h) * p.Ns + js] = make_uint4(w[4 * h], w[4 * h + 1], w[4 * h + 2], w[4 * h + 3]);
    if (off) oq[q] = make_uint4(o[0], o[1], o[2], o[3]);
}

// The four lanes l, l + 16, l + 32, l + 48 of a wave share a source, each over a quarter of the
// receivers (the quarters' ring rows start 16 LDS banks apart, so their reads of one step's
// few consecutive slots meet in different banks). Up to GPW far groups per wave. R ring slots
// (time mod R) per receiver, the first PITCH - R repeated after the last so that a run of
// slots never wraps. NT slots per near sum, t + 2 - NT .. t + 1. Near and far operands have
// their own registers, filled from L2 in chunks of 16 receivers, each register refilled with the
// following chunk's as soon as it is used.
// The first waves of a workgroup (p.nwg of them, 4 to 14) do the sums, the others (1 to 4) run
// NPL neurons per lane: roles of their own, so that neither holds the other's registers. A step:
// near sums | barrier | far sums, beside the neurons | barrier.
template <int GPW, int NPL, bool WBF, bool OFF, int R, int PITCH, int NT>
__global__ void __launch_bounds__(1024) hyb_block_bwd_kernel(HybBlk p) {
    extern __shared__ float smem[];
    // (OFF) what the caller stated does not hold: the general scan, launched behind this one,
    // takes the call, or every output becomes NaN
    const bool wrong = OFF && *p.wrong != 0;
    if (wrong && p.wt) return;
    constexpr int WV = WBF ? 2 : 4;                        // uint4 of W per chunk
    constexpr int CPW = 16 / WV;                           // receivers per uint4 of W
    constexpr uint32_t MB = R * 4 - 1;                     // byte offset within the R slots
    constexpr int PAD = R <= 16 ? 16 : 32;                 // words between the quarters
    constexpr int PF = 2;                                  // steps of gy / u loaded ahead
    static_assert(NT <= PITCH - R + 1 && PITCH - R >= 3, "runs of slots past the repeated ones");
    const int N = p.N, T = p.T, B = p.B, Ns = p.Ns, NCl = p.NCl, RG = p.RG;
    const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = p.nwg;   // waves that sum
    const int part = lane >> 4, src = lane & 15;
    const int ngroups = (N + 15) >> 4;
    const float sv = p.s_uniform;
    const int omin = p.meta ? p.meta[1] : 0;
    auto lag_of = [&](int j) {                             // (one offset: taps below lag 1 are dropped)
        const int l = first_lag(1.0f + p.base[j], sv) + omin;
        return OFF ? l : max(l, 1);
    };
    // groups in first-lag order: near ones first
    const int glo = tid < ngroups ? lag_of(p.order[tid * 16]) : 0x7fffffff;
    const int nn = __syncthreads_count(glo < 4);

    const int rowsq = NCl * 16 * PITCH + PAD;              // words per quarter
    float* ghist = smem + 4 * rowsq + 64;                  // [RG][Ns], column = source
    float* npart = ghist + (size_t)RG * Ns;                // near partials [group][slice][NT][16]
    for (int q = tid; q < 4 * rowsq + 64 + RG * Ns + p.room; q += blockDim.x) smem[q] = 0.0f;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float*)smem;
    const uint32_t rowb = lds0 + (uint32_t)(part * rowsq) * 4u;   // the lane's first receiver row

    // near groups: 1, 2 or 4 slices of the receivers, as many as the partials' room, the chunks and
    // the waves allow; units (group, slice) dealt out to the waves
    int slices = 4;
    while (slices > 1 && (slices > NCl || nn * slices * NT * 16 > p.room || nn * slices >= 2 * nw)) slices >>= 1;
    const int per_slice = (NCl + slices - 1) / slices;
    const int units = nn * slices;

    // this wave's far groups, and those of blocks of 4 steps among them
    auto far_group = [&](int q) { return nn + ((q & 1) ? (q + 1) * nw - 1 - wave : q * nw + wave); };
    int nfar = 0;
    uint32_t longer = 0;
    int jf[GPW];
#pragma unroll
    for (int q = 0; q < GPW; ++q) {
        const int g = far_group(q);
        jf[q] = g * 16 + src < N ? p.order[g * 16 + src] : -1;
        if (g < ngroups) {
            nfar = q + 1;
            longer |= (lag_of(p.order[g * 16]) >= 8 ? 1u : 0u) << q;
        }
    }
    nfar = __builtin_amdgcn_readfirstlane(nfar);
    longer = __builtin_amdgcn_readfirstlane(longer);
    // chunks per step of a block of 4 and of 2 steps
    const int ch4 = (NCl + 3) >> 2, ch2 = (NCl + 1) >> 1;
    auto far_first = [&](int q, int t) { return ((longer >> q) & 1) ? (3 - (t & 3)) * ch4 : (1 - (t & 1)) * ch2; };

    const i32x4 rw = buffer_rsrc(p.wq, (uint32_t)((size_t)4 * NCl * WV * Ns * 16));
    const i32x4 ro = buffer_rsrc(p.oq, OFF ? (uint32_t)((size_t)4 * NCl * Ns * 16) : 0u);
    const int wl = (part * NCl * WV * Ns + src) * 16, ol = (part * NCl * Ns + src) * 16;
    auto load4 = [](i32x4 rs, int voff, int soff) {
        const i32x4 v = raw_buffer_load_i32x4(rs, voff, soff, 0);
        return make_uint4((uint32_t)v.x, (uint32_t)v.y, (uint32_t)v.z, (uint32_t)v.w);
    };
    // the operands of the next chunk to sum
    struct Chunk { uint4 w[WV], o; };
    constexpr bool DEEP = GPW > 1 && !OFF;                 // registers for a second chunk of each
    Chunk nearc, nears, farc, fars;
    auto fetch_w = [&](Chunk& ch, int h, int gb, int c) { ch.w[h] = load4(rw, wl, ((c * WV + h) * Ns + gb) * 16); };
    auto fetch_o = [&](Chunk& ch, int gb, int c) {
        if constexpr (OFF) ch.o = load4(ro, ol, (c * Ns + gb) * 16);
    };
    auto fetch = [&](Chunk& ch, int gb, int c) {
#pragma unroll
        for (int h = 0; h < WV; ++h) fetch_w(ch, h, gb, c);
        fetch_o(ch, gb, c);
    };

    // acc[n] += sum over chunk c's 16 receivers of W gr(slot + n), slot byte st; then (refill) the
    // operands of chunk nc of the group at source slot ngb come in
    auto sum_chunk = [&](Chunk& ch, int c, uint32_t st, bool refill, int ngb, int nc, auto& acc) {
        constexpr int NP = sizeof(acc) / sizeof(float);
        constexpr int GR = NP >= 4 ? 2 : 4;                // receivers read together
        const uint32_t cb = rowb + (uint32_t)c * (16 * PITCH * 4);
        if constexpr (!OFF) {
            // every source reads the same slots: lane `src` reads receiver src's, and each
            // multiply-add takes its receiver's value from that lane of the row
            float g[NP];
            const auto* x = (const __attribute__((address_space(3))) float*)(uintptr_t)(cb + st + (uint32_t)src * (PITCH * 4));
#pragma unroll
            for (int n = 0; n < NP; ++n) g[n] = x[n];
            auto four = [&](auto e0) {                     // receivers E .. E + 3
                constexpr int E = decltype(e0)::value;
                float wf[4];
                if constexpr (WBF) {
                    const uint4& v = ch.w[E >> 3];
                    const uint32_t a = E & 4 ? v.z : v.x, b2 = E & 4 ? v.w : v.y;
                    wf[0] = __uint_as_float(a << 16); wf[1] = __uint_as_float(a & 0xFFFF0000u);
                    wf[2] = __uint_as_float(b2 << 16); wf[3] = __uint_as_float(b2 & 0xFFFF0000u);
                } else {
                    const uint4& v = ch.w[E >> 2];
                    wf[0] = __uint_as_float(v.x); wf[1] = __uint_as_float(v.y);
                    wf[2] = __uint_as_float(v.z); wf[3] = __uint_as_float(v.w);
                }
                add_rows<E>(wf, g, acc);
                if ((E + 4) % CPW == 0 && refill) fetch_w(ch, E / CPW, ngb, nc);
            };
            four(std::integral_constant<int, 0>{});
            four(std::integral_constant<int, 4>{});
            four(std::integral_constant<int, 8>{});
            four(std::integral_constant<int, 12>{});
            return;
        }
        // four slots of connections at a time: no byte carries over (both summands < 128)
        uint4 oc = make_uint4(st, st, st, st);
        if constexpr (OFF) {
            constexpr uint32_t M4 = MB * 0x01010101u;
            const uint32_t s4 = st * 0x01010101u;
            oc = make_uint4((ch.o.x + s4) & M4, (ch.o.y + s4) & M4, (ch.o.z + s4) & M4, (ch.o.w + s4) & M4);
            if (refill) fetch_o(ch, ngb, nc);
        }
        float r[2][GR][NP];
        auto read = [&](int e0, float (&v)[GR][NP]) {
#pragma unroll
            for (int q = 0; q < GR; ++q) {
                const int e = e0 + q;
                const uint32_t ow = e < 4 ? oc.x : e < 8 ? oc.y : e < 12 ? oc.z : oc.w;
                const uint32_t a = cb + (OFF ? (ow >> (8 * (e & 3))) & 0xFFu : ow);
                const auto* x = (const __attribute__((address_space(3))) float*)(uintptr_t)a + e * PITCH;
#pragma unroll
                for (int n = 0; n < NP; ++n) v[q][n] = x[n];
            }
        };
        read(0, r[0]);
#pragma unroll
        for (int e0 = 0; e0 < 16; e0 += GR) {
            const int cur = (e0 / GR) & 1;
            if (e0 + GR < 16) read(e0 + GR, r[cur ^ 1]);
#pragma unroll
            for (int q = 0; q < GR; ++q) {
                const int e = e0 + q;
                float wv;
                if constexpr (WBF) {
                    const uint4& x = ch.w[e >> 3];
                    const int e8 = e & 7;
                    const uint32_t w2 = e8 < 2 ? x.x : e8 < 4 ? x.y : e8 < 6 ? x.z : x.w;
                    wv = __uint_as_float((e & 1) ? (w2 & 0xFFFF0000u) : (w2 << 16));
                } else {
                    const uint4& x = ch.w[e >> 2];
                    const int e4 = e & 3;
                    wv = __uint_as_float(e4 == 0 ? x.x : e4 == 1 ? x.y : e4 == 2 ? x.z : x.w);
                }
#pragma unroll
                for (int n = 0; n < NP; ++n) acc[n] = fmaf(wv, r[cur][q][n], acc[n]);
            }
            if ((e0 + GR) % CPW == 0 && refill) fetch_w(ch, (e0 + GR) / CPW - 1, ngb, nc);
            __builtin_amdgcn_sched_barrier(0);             // bounds the reads in flight (registers)
        }
    };
    auto quarters = [](float v) {
        v += __shfl_xor(v, 16);
        return v + __shfl_xor(v, 32);
    };

    const size_t BN = (size_t)B * N;
    const int tend = p.gz ? -4 : 0;                        // gz: the blocks that reach step 0
    auto keep_gz = [&](int tau, int j, float v) {
        if (p.gz && tau >= 0 && tau < T) p.gz[(size_t)tau * BN + (size_t)b * N + j] = v;
    };
    if (wave >= nw) {
        // ---- neurons
        const Lif k = p.lif;
        const uint32_t row_bytes = (uint32_t)BN * 4u;
        const float is2 = 1.0f / (sv * sv);
        const uint32_t lags = (uint32_t)(p.L - 1);         // of the window: 1 .. L - 1
        int jn[NPL], lon[NPL], voff[NPL];
        float m[NPL], cn[NPL], x0[NPL], lam[NPL], dbacc[NPL];
        float* own[NPL];
        const float* mine[NPL];
        bool near_j[NPL];
#pragma unroll
        for (int i = 0; i < NPL; ++i) {
            const int jt = (wave - nw + i * ((int)(blockDim.x >> 6) - nw)) * 64 + lane;
            const bool act = jt < N;
            const int j = act ? jt : 0;
            jn[i] = act ? j : -1;
            voff[i] = act ? (b * N + j) * 4 : kOutOfRange;
            m[i] = p.drop ? p.drop[(size_t)b * N + j] : 1.0f;
            cn[i] = 1.0f + p.base[j];
            const int lob = first_lag(cn[i], sv);          // before the offset
            lon[i] = lob + omin;
            x0[i] = (float)lob - cn[i];                    // (exact)
            own[i] = smem + (j / (NCl * 16)) * rowsq + (j % (NCl * 16)) * PITCH;
            const int slot = p.rank[j];
            near_j[i] = act && slot < nn * 16;
            mine[i] = npart + (slot < nn * 16 ? (slot >> 4) * slices * NT * 16 + (slot & 15) : 0);
            lam[i] = 0.0f;
            dbacc[i] = 0.0f;
        }
        auto at_step = [&](const float* x, int t) {
            return step_rsrc((uint64_t)x + (uint64_t)max(t, 0) * row_bytes, t >= 0 ? row_bytes : 0u);
        };
        // gy and u of PF steps in registers while the next PF steps' load (a rotation by one step
        // would wait for the newest load in every step)
        float gq[NPL][PF], uq[NPL][PF], gn[NPL][PF], un[NPL][PF];
        auto load_steps = [&](int t, float (&g)[NPL][PF], float (&u)[NPL][PF]) {
#pragma unroll
            for (int q = 0; q < PF; ++q) {
#pragma unroll
                for (int i = 0; i < NPL; ++i) {
                    g[i][q] = raw_buffer_load_f32(at_step(p.gy, t - q), voff[i], 0, 0);
                    u[i][q] = raw_buffer_load_f32(at_step(p.u, t - q), voff[i], 0, 0);
                }
            }
        };
        load_steps(T - 1, gq, uq);
        __builtin_amdgcn_s_setprio(3);                     // the step waits for this chain
        int g1 = T % RG;                                   // (t + 1) mod RG
        __syncthreads();
        for (int t = T - 1; t >= tend; --t) {
            const int r = (T - 1 - t) & (PF - 1);
            const bool live = t >= 0;
            if (r == 0) load_steps(t - PF, gn, un);
            barrier_lds();
            // near sources' sums, and below lag 1 the taps on the truncated ones (all the lane's
            // neurons at each stage: one LDS round trip for all of them)
            float v[NPL][NT][4], gfs[NPL], gnear[NPL];
#pragma unroll
            for (int i = 0; i < NPL; ++i)
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                    for (int q = 0; q < 4; ++q) v[i][n][q] = mine[i][((q < slices ? q : 0) * NT + n) * 16];
#pragma unroll
            for (int i = 0; i < NPL; ++i) {
                gfs[i] = 0.0f;
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    float a = v[i][n][0];
#pragma unroll
                    for (int q = 1; q < 4; ++q) a += q < slices ? v[i][n][q] : 0.0f;
                    if (n < NT - 1)
                        gfs[i] = fmaf(fmaxf(sv - fabsf((float)(n + 2 - NT - omin) - cn[i]), 0.0f), near_j[i] ? a : 0.0f, gfs[i]);
                    gnear[i] = a;
                }
            }
#pragma unroll
            for (int i = 0; i < NPL; ++i)
                if (near_j[i]) ghist[__umul24(g1, Ns) + jn[i]] = gnear[i];
            // (four taps at a time: the weights are formed here and not held in registers; a tap past
            // the triangle weighs 0)
#pragma unroll 1
            for (int f0 = 0; f0 < p.KF; f0 += 4) {
                float gv[NPL][4];
#pragma unroll
                for (int i = 0; i < NPL; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        int sl = g1 + min(max(lon[i] + f0 + q, 1), RG - 1) - 1;   // (outside the window: unused)
                        sl = sl >= RG ? sl - RG : sl;
                        gv[i][q] = ghist[__umul24(sl, Ns) + max(jn[i], 0)];
                    }
#pragma unroll
                for (int i = 0; i < NPL; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float h = fmaxf(sv - fabsf(x0[i] + (float)(f0 + q)), 0.0f);
                        gfs[i] = fmaf((uint32_t)(lon[i] + f0 + q - 1) < lags ? h : 0.0f, gv[i][q], gfs[i]);
                    }
            }
#pragma unroll
            for (int i = 0; i < NPL; ++i) {
                if (near_j[i]) keep_gz(t + 1, jn[i], gnear[i]);
                float gf = gfs[i];
                gf *= is2;
                const float u = r == 0 ? uq[i][0] : uq[i][1], gyv = r == 0 ? gq[i][0] : gq[i][1];
                const float y = lif_fire(k, u);
                const float du = lif_backward(k, gyv + gf, u, y, lam[i]);
                lam[i] = k.decay * du;
                const float da = wrong ? __builtin_nanf("") : lif_dx(k, du);
                const float gr = da * m[i];
                if (jn[i] >= 0 && !wrong) {
                    const int sw = t & (R - 1);
                    own[i][sw] = live ? gr : 0.0f;
                    if (sw < PITCH - R) own[i][sw + R] = live ? gr : 0.0f;
                    if (NT > 1) {                          // the early slot that step t - 1 reads first
                        const int sz = (t - NT + 1) & (R - 1);
                        own[i][sz] = 0.0f;
                        if (sz < PITCH - R) own[i][sz + R] = 0.0f;
                    }
                }
                raw_buffer_store_f32(da, at_step(p.dx, t), voff[i], 0, 0);
                if (p.gr) raw_buffer_store_f32(gr, at_step(p.gr, t), voff[i], 0, 0);
                dbacc[i] += live ? gr : 0.0f;
            }
            if (r == PF - 1) {
#pragma unroll
                for (int i = 0; i < NPL; ++i)
#pragma unroll
                    for (int q = 0; q < PF; ++q) {
                        gq[i][q] = gn[i][q];
                        uq[i][q] = un[i][q];
                    }
            }
            barrier_lds();
            g1 = g1 == 0 ? RG - 1 : g1 - 1;
        }
#pragma unroll
        for (int i = 0; i < NPL; ++i)
            if (jn[i] >= 0) p.part[(size_t)b * N + jn[i]] = dbacc[i];
        return;
    }

    // ---- sums
    int g1 = T % RG;                                       // (t + 1) mod RG
    float acc[GPW][4];                                     // far blocks under way
#pragma unroll
    for (int q = 0; q < GPW; ++q)
#pragma unroll
        for (int n = 0; n < 4; ++n) acc[q][n] = 0.0f;
    // the wave's first near unit; whether it is all its near work, one chunk or two: it stays loaded
    const int u_gb = wave / slices * 16, u_c = min(wave % slices * per_slice, NCl - 1);
    const bool one = per_slice <= (DEEP ? 2 : 1) && wave + nw >= units;
    const bool both = per_slice == 2 && u_c + 1 < NCl;
    if (wave < units) fetch(nearc, u_gb, u_c);
    if (DEEP && wave < units && both) fetch(nears, u_gb, u_c + 1);
    if (nfar > 0) {
        const int c = min(far_first(0, T - 1), NCl - 1);
        fetch(farc, far_group(0) * 16, c);
        if constexpr (DEEP) fetch(fars, far_group(0) * 16, min(c + 1, NCl - 1));
    }
    __syncthreads();
    for (int t = T - 1; t >= tend; --t) {
        for (int u = wave; u < units; u += nw) {
            float cur[NT];
#pragma unroll
            for (int n = 0; n < NT; ++n) cur[n] = 0.0f;
            const uint32_t st = ((uint32_t)(t + 2 - NT) * 4u) & MB;
            if (one) {
                if (wave % slices * per_slice < NCl) {
                    sum_chunk(nearc, u_c, st, false, 0, 0, cur);
                    if constexpr (DEEP) {
                        if (both) sum_chunk(nears, u_c + 1, st, false, 0, 0, cur);
                    }
                }
            } else {
                const int g = u / slices, sl = u - g * slices;
                const int c0 = min(sl * per_slice, NCl), c1 = min(c0 + per_slice, NCl);
                const int un1 = u + nw < units ? u + nw : wave, gx = un1 / slices;
                const int cx = min((un1 - gx * slices) * per_slice, NCl - 1);
#pragma unroll 1
                for (int c = c0; c < c1; ++c) {
                    const bool last = c + 1 == c1;
                    sum_chunk(nearc, c, st, true, (last ? gx : g) * 16, last ? cx : c + 1, cur);
                }
                if (c0 >= c1) fetch(nearc, gx * 16, cx);   // (a slice past the last chunk)
            }
            float* o = npart + (size_t)u * NT * 16 + src;
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                const float a = quarters(cur[n]);
                if (part == 0) o[n * 16] = a;
            }
        }
        barrier_lds();
        // far sums: slots t + 1 and later only
#pragma unroll 1
        for (int q = 0; q < nfar; ++q) {
            const bool p4 = (longer >> q) & 1;
            const int P = p4 ? 4 : 2, sub = P - 1 - (t & (P - 1));
            const int c0 = far_first(q, t), c1 = c0 + (p4 ? ch4 : ch2);
            const uint32_t st = ((uint32_t)(t + 1 + sub) * 4u) & MB;
            // what follows: the next far group, or the first one in the next step
            const int qx = q + 1 < nfar ? q + 1 : 0;
            const int gx = far_group(qx) * 16, cx = min(far_first(qx, q + 1 < nfar ? t : t - 1), NCl - 1);
            float cur[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (sub != 0) {
#pragma unroll
                for (int x = 0; x < GPW; ++x)
                    if (x == q) {
#pragma unroll
                        for (int n = 0; n < 4; ++n) cur[n] = acc[x][n];
                    }
            }
            auto sum_far = [&](Chunk& ch, int c, int ngb, int nc) {
                if (c >= NCl) {                            // (the last step of a block may have fewer)
                    fetch(ch, ngb, min(nc, NCl - 1));
                } else if (p4) {
                    sum_chunk(ch, c, st, true, ngb, min(nc, NCl - 1), cur);
                } else {
                    float (&c2)[2] = reinterpret_cast<float (&)[2]>(cur);
                    sum_chunk(ch, c, st, true, ngb, min(nc, NCl - 1), c2);
                }
            };
            if constexpr (DEEP) {                          // chunks in pairs, the next pair on its way
#pragma unroll 1
                for (int c = c0; c < c1; c += 2) {
                    const bool last = c + 2 >= c1;
                    const int ngb = last ? gx : far_group(q) * 16, nc = last ? cx : c + 2;
                    sum_far(farc, c, ngb, nc);
                    if (c + 1 < c1) sum_far(fars, c + 1, ngb, nc + 1);
                    else if (last) fetch(fars, ngb, min(nc + 1, NCl - 1));
                }
            } else {
#pragma unroll 1
                for (int c = c0; c < c1; ++c) {
                    const bool last = c + 1 == c1;
                    sum_far(farc, c, last ? gx : far_group(q) * 16, last ? cx : c + 1);
                }
            }
            if (sub != P - 1) {
#pragma unroll
                for (int x = 0; x < GPW; ++x)
                    if (x == q) {
#pragma unroll
                        for (int n = 0; n < 4; ++n) acc[x][n] = cur[n];
                    }
                continue;
            }
            // the block is whole: G(t + P .. t + 2 P - 1)
            int js = -1;
#pragma unroll
            for (int x = 0; x < GPW; ++x) js = x == q ? jf[x] : js;
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                if (n < P) {
                    const float a = quarters(cur[n]);
                    int sl = g1 + P + n - 1;
                    sl = sl >= RG ? sl - RG : sl;
                    if (part == 0 && js >= 0) {
                        ghist[__umul24(sl, Ns) + js] = a;
                        keep_gz(t + P + n, js, a);
                    }
                }
            }
        }
        barrier_lds();
        g1 = g1 == 0 ? RG - 1 : g1 - 1;
    }
}

namespace {

template <int GPW, int NPL, bool WBF, bool OFF, int R, int PITCH, int NT>
bool launch_one(const HybBlk& p, const HybBlkShape& q, hipStream_t s) {
    const auto fn = hyb_block_bwd_kernel<GPW, NPL, WBF, OFF, R, PITCH, NT>;
    ensure_lds((const void*)fn, q.lds);
    hipLaunchKernelGGL(fn, dim3(p.B), dim3(q.block), q.lds, s, p);
    return true;
}

template <int GPW, int NPL, bool WBF>
bool launch_ring(const HybBlk& p, const HybBlkShape& q, hipStream_t s) {
    if (!p.oq) {
        if constexpr (GPW > 1) return launch_one<GPW, NPL, WBF, false, 8, 12, 1>(p, q, s);
        return false;
    }
    if (q.R == 32) return launch_one<GPW, NPL, WBF, true, 32, 40, 8>(p, q, s);
    if (q.NT == 1) return launch_one<GPW, NPL, WBF, true, 16, 20, 1>(p, q, s);
    if (q.NT == 2) return launch_one<GPW, NPL, WBF, true, 16, 20, 2>(p, q, s);
    return launch_one<GPW, NPL, WBF, true, 16, 20, 4>(p, q, s);
}

}  // namespace

HybBlkShape hyb_block_shape(int N, int L, bool bf16, bool offsets, int D, int KF, int NT, size_t max_lds) {
    HybBlkShape q{};
    if (N < 1 || N > 1024 || D < 1 || KF < 1 || KF > kTapsMax || NT > 8) return q;
    // steps whose slots must differ: t - NT + 1 (early run) .. t + 7 (spread block of 4 steps) and
    // the D - 1 offsets
    q.R = !offsets ? 8 : 6 + NT + D <= 16 && NT <= 4 ? 16 : 6 + 8 + D <= 32 ? 32 : 0;
    if (!q.R) return q;
    q.NT = q.R <= 16 ? NT : 8;
    q.Dmax = q.R - 6 - q.NT;
    const int groups = (N + 15) / 16;
    q.NPL = N <= 192 ? 1 : N <= 384 ? 2 : 4;
    q.NCl = (N + 63) / 64;
    const int neuron_waves = (N + 64 * q.NPL - 1) / (64 * q.NPL);
    q.nwg = std::min(16 - neuron_waves, std::max(groups * std::min(q.NCl, 4), 4));   // far groups per wave: at most 1, 2, 3, 6 (N <= 192, 384, 512, 1024)
    q.block = (q.nwg + neuron_waves) * 64;
    q.Ns = groups * 16;
    q.RG = std::max(L, 8) + 1;                             // steps t + 1 .. t + L - 1, blocks to t + 7
    const int pitch = q.R == 8 ? 12 : q.R == 16 ? 20 : 40, pad = q.R <= 16 ? 16 : 32;
    const size_t words = (size_t)4 * (q.NCl * 16 * pitch + pad) + 64 + (size_t)q.RG * q.Ns;
    // near partials: one slice of every group at least, up to 16 KB
    const size_t least = (size_t)q.Ns * q.NT;
    q.wq = (size_t)4 * q.NCl * (bf16 ? 2 : 4) * q.Ns;
    q.oq = offsets ? (size_t)4 * q.NCl * q.Ns : 0;
    const size_t avail = max_lds / sizeof(float);
    if (words + least > avail || (!offsets && N <= 256)) return q;
    q.room = (int)std::min(avail - words, std::max(least, (size_t)4096));
    q.lds = (words + q.room) * sizeof(float);
    q.ok = true;
    return q;
}

void launch_hyb_block_pack(const HybBlk& p, const HybBlkShape& q, uint4* wq, uint4* oq, int* order, const void* W,
                           const int8_t* off, bool bf16, hipStream_t s) {
    hipLaunchKernelGGL(hyb_block_order_kernel, dim3(1), dim3(1024), 0, s, p.base, p.s_uniform, p.N, p.meta, q.NT,
                       q.Dmax, order, order + p.N, order + 2 * p.N);
    const int blocks = (4 * p.NCl * p.Ns + 255) / 256;
    if (bf16) hipLaunchKernelGGL(hyb_block_pack_kernel<true>, dim3(blocks), dim3(256), 0, s, p, wq, oq, W, off);
    else hipLaunchKernelGGL(hyb_block_pack_kernel<false>, dim3(blocks), dim3(256), 0, s, p, wq, oq, W, off);
}

bool launch_hyb_block_bwd(const HybBlk& p, const HybBlkShape& q, bool bf16, hipStream_t s) {
    if (p.N <= 192) return bf16 ? launch_ring<1, 1, true>(p, q, s) : launch_ring<1, 1, false>(p, q, s);
    if (p.N <= 384) return bf16 ? launch_ring<2, 2, true>(p, q, s) : launch_ring<2, 2, false>(p, q, s);
    if (p.N <= 512) return bf16 ? launch_ring<3, 4, true>(p, q, s) : launch_ring<3, 4, false>(p, q, s);
    return bf16 ? launch_ring<6, 4, true>(p, q, s) : launch_ring<6, 4, false>(p, q, s);
}

}  // namespace delrec
