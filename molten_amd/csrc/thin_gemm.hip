// thin_gemm.hip -- Q4 products on two or three workgroups per CU: the grouped
// GEMMs of the prefill step (over launch-ordered maps) and the dense prefill
// projections.
//
// Same products as grouped_gemm.hip's segment kernel, bit for bit: the MFMAs
// of an output run over k in the same order.  With few rows per expert they
// are bound by reading every chosen expert's weights (5.3 MB each) and turning
// their codes into bf16 (19 VALU instructions per 8 codes), with many by the
// matrix cores.  A lone wave issues a VALU instruction every ~5 cycles where a
// SIMD takes one every 2 to 4, so the tile gives up rows for waves: at most
// four row blocks of 32 per pass in 80 KB of LDS and 256 registers, two
// workgroups per CU (three with one row block), whose loads, dequant and
// MFMAs cover each other.  That pays for dequantizing an expert's codes once
// per 128 rows instead of once per 288.  A column's scales and biases are read
// whole into registers, 64 bytes of a row at a time.
//
// Gate/up and down of 64 experts (2048 x 1536, top-4), 100 tokens: 57.6 + 31.0
// us, 215 + 108 MB fetched (the segment kernel 97 + 50 us, 225 + 112 MB); 4096
// tokens 220 + 117 us at best, 593 + 296 MB (225 + 126 us, 367 + 184 MB): the
// passes of an expert fetch its codes again.  Dense 4095 x 6144 x 2048: 93 us
// (1110 TFLOP/s; the segment kernel 116), 1023 x 6144 x 2048 35 (60).
#include <algorithm>

#include "mh_device.hpp"
#include "mh_host.hpp"
#include "mh_q4gemm.hpp"

namespace {

using namespace mh;

constexpr int kThinWaves = 4;
constexpr int kThinJ = 4;  // scale blocks of 512 k held in registers

// LDS of a workgroup: A in NSA slots of 64 k, and per wave two slots of B
// codes (128 k of NB column blocks).
template <int RBMAX, int NB>
struct ThinLayout {
    static constexpr int NSA = 3;
    static constexpr int A_SLOT = RBMAX * 32 * 128;
    static constexpr int B_SLOT = kThinWaves * NB * 2048;
    static constexpr int B_OFF = NSA * A_SLOT;
    static constexpr int LDS = B_OFF + 2 * B_SLOT;
    static constexpr int WGS = LDS <= 160 * 1024 / 3 ? 3 : 2;  // workgroups per CU
    static_assert(LDS <= 80 * 1024, "two workgroups per CU");
};

// One pass: rows [mp0, mp0 + 32 RB) of the segment, the wave's NB column
// blocks, the whole K in stages of 64 (four MFMA steps), unrolled over the 8
// stages of a scale block.
//
// A arrives by direct-to-LDS loads shared by the workgroup, NSA stages ahead
// (a slot is refilled after the barrier that ends its stage); chunk c (16
// bytes) of row r sits at chunk c ^ ((r >> 1) & 7) of its 128-byte row, so
// that 16 lanes reading one chunk of 16 rows cover all 64 banks.  Codes and
// scales come into regions of the wave's own, so they need no barrier: a
// stage's codes are read into registers before it starts, and a code slot is
// refilled, two blocks ahead, as soon as its second half is read; the scale
// words of 512 k are read at once.  The loads of a wave complete in issue
// order, so the one wait per stage is a count of what was issued after the
// next stage's A.
template <int RB, int RBMAX, int NBW, int NMAT, bool GATHER, int EPI>
__device__ __forceinline__ void thin_pass(const GemmArgs& a, uint32_t brow, uint32_t n0, uint32_t mp0,
                                          uint32_t m_end, uint32_t lds0, int lane_in, int wave) {
    constexpr int NB = NMAT * NBW;
    using L = ThinLayout<RBMAX, NB>;
    constexpr int NSA = L::NSA;
    constexpr int QA = RB;                    // A loads (1 KB) per wave per stage
    // recomputed in every pass (hoisted out of the pass loop they cost registers)
    const int lane = static_cast<int>(opaque(static_cast<uint32_t>(lane_in)));
    const int i32 = lane & 31, h = lane >> 5;
    const uint32_t K = a.k, groups = K / 64u;
    const uint32_t nj = K / 512u;             // scale blocks (8 stages, 4 code blocks each)

    const gbytes abase = uniform_ptr(a.a);
    gbytes cbase[NMAT], sbase[NMAT], bbase[NMAT];
    cbase[0] = uniform_ptr(a.c0);
    sbase[0] = uniform_ptr(a.s0);
    bbase[0] = uniform_ptr(a.b0);
    if (NMAT == 2) {
        cbase[NMAT - 1] = uniform_ptr(a.c1);
        sbase[NMAT - 1] = uniform_ptr(a.s1);
        bbase[NMAT - 1] = uniform_ptr(a.b1);
    }
    uint32_t aoffs[QA];
#pragma unroll
    for (int q = 0; q < QA; ++q) {
        const uint32_t r = 8u * (wave * QA + q) + static_cast<uint32_t>(lane >> 3);
        const uint32_t m = min(mp0 + r, m_end - 1u);
        uint32_t src = GATHER ? a.gather[m] : m;
        src = min(src, a.a_rows - 1u);
        const uint32_t chunk = static_cast<uint32_t>(lane & 7) ^ ((r >> 1) & 7u);
        aoffs[q] = src * K * 2u + chunk * 16u;
    }
    // codes: load p of fragment t fills columns 16p .. 16p + 15 (4 lanes of 16
    // bytes each, chunk g at position g ^ ((column >> 2) & 3)); scales and
    // biases: lane (i32, h) loads 16 bytes of column i32's scales or biases
    uint32_t bcoffs[NB][2], sboff[NB];
#pragma unroll
    for (int cb = 0; cb < NBW; ++cb) {
#pragma unroll
        for (int mat = 0; mat < NMAT; ++mat) {
            const int t = mat * NBW + cb;
            const uint32_t col0 = brow + static_cast<uint32_t>((wave * NBW + cb) * 32);
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const uint32_t c = 16u * p + static_cast<uint32_t>(lane >> 2);
                const uint32_t r = min(col0 + c, a.w_rows - 1u);
                const uint32_t g = static_cast<uint32_t>(lane & 3) ^ ((c >> 2) & 3u);
                bcoffs[t][p] = r * (K / 2u) + g * 16u;
            }
            sboff[t] = min(col0 + static_cast<uint32_t>(i32), a.w_rows - 1u) * groups * 2u;
        }
    }
    // the column's scales (lanes 0-31) and biases (lanes 32-63), 512 k an
    // element: kThinJ scale blocks from block j on
    uint4 sbr[NB][kThinJ];
    auto load_sb = [&](uint32_t j) {
#pragma unroll
        for (int t = 0; t < NB; ++t) {
            const gbytes src = (h ? bbase[t / NBW] : sbase[t / NBW]) + sboff[t];
#pragma unroll
            for (int i = 0; i < kThinJ; ++i) {
                const u32x4 v = *reinterpret_cast<const __attribute__((address_space(1))) u32x4*>(
                    src + min(j + i, nj - 1u) * 16u);
                sbr[t][i] = make_uint4(v.x, v.y, v.z, v.w);
            }
        }
    };
    load_sb(0);
    auto issue_a = [&](uint32_t s) {
        const uint32_t buf = __builtin_amdgcn_readfirstlane(lds0 + (s % NSA) * L::A_SLOT + wave * QA * 1024u);
        const gbytes ag = uniform_ptr(abase + s * 128u);
        static_for<QA>([&](auto q) { dma16m<q * 1024>(ag, aoffs[q], buf); });
    };
    auto issue_b = [&](uint32_t b, auto slot_c) {  // code block b into its slot (b % 2)
        const uint32_t buf = __builtin_amdgcn_readfirstlane(lds0 + L::B_OFF + decltype(slot_c)::value * L::B_SLOT + wave * NB * 2048u);
        static_for<NB>([&](auto t) {
            const gbytes cg = uniform_ptr(cbase[t / NBW] + b * 64u);
            dma16m<t * 2048>(cg, bcoffs[t][0], buf);
            dma16m<t * 2048 + 1024>(cg, bcoffs[t][1], buf);
        });
    };
    f32x16_t acc[NMAT][RB][NBW];
#pragma unroll
    for (int mat = 0; mat < NMAT; ++mat)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int cb = 0; cb < NBW; ++cb)
#pragma unroll
                for (int q = 0; q < 16; ++q) acc[mat][rb][cb][q] = 0.0f;

    // LDS reads (no wait): the code chunk of stage u of a scale block (chunk
    // 2 (u % 2) + h of the lane's column), a scale block's words, A fragments
    const uint32_t bswz = (static_cast<uint32_t>(i32) >> 2) & 3u;
    uint32_t bat[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        bat[u] = lds0 + L::B_OFF + wave * NB * 2048u + i32 * 64u + ((2u * u + static_cast<uint32_t>(h)) ^ bswz) * 16u;
    }
    auto read_b = [&](auto u_c, uint4 (&bc)[NB]) {
        constexpr int u = decltype(u_c)::value;
        static_for<NB>([&](auto t) { bc[t] = lds_read16_at<((u / 2) & 1) * L::B_SLOT + t * 2048>(bat[u & 1]); });
    };
    uint32_t aoff[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        aoff[j] = static_cast<uint32_t>(i32) * 128u +
                  ((static_cast<uint32_t>(4 * h + j) ^ ((static_cast<uint32_t>(i32) >> 1) & 7u)) * 16u);
    }
    auto read_a = [&](uint32_t s, int j, uint4 (&av)[RB]) {
        const uint32_t at = lds0 + (s % NSA) * L::A_SLOT + aoff[j];
        static_for<RB>([&](auto rb) { av[rb] = lds_read16_at<rb * 4096>(at); });
    };
    float sf[NB], bf[NB];
    auto word = [](const uint4& v, int j) { return j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w; };
    // scales and biases of stage u: at even stages the word of both its group
    // and the next's is spread from the lane half that holds it
    uint32_t sw[NB], bw[NB];
    auto scale_bias = [&](int u) {
#pragma unroll
        for (int t = 0; t < NB; ++t) {
            if ((u & 1) == 0) {
                const uint32_t x = word(sbr[t][0], u / 2);
                const auto both = __builtin_amdgcn_permlane32_swap(x, x, false, false);
                sw[t] = both[0];
                bw[t] = both[1];
            }
            sf[t] = __uint_as_float((u & 1) ? sw[t] & 0xffff0000u : sw[t] << 16);
            bf[t] = __uint_as_float((u & 1) ? bw[t] & 0xffff0000u : bw[t] << 16);
        }
    };

    uint4 bc[NB];
    uint4 av[2][RB];
    bf16x8_t bfr[2][NB];
    using c0 = std::integral_constant<int, 0>;
    using c1 = std::integral_constant<int, 1>;
    // issue order as in the loop: a stage's A, then the codes issued before
    // the A of the stages after it
    issue_b(0, c0{});
    issue_a(0);
    issue_a(1);
    issue_b(1, c1{});
    issue_a(2);
    wait_vmcnt<0>();  // (the compiler waits for the scales by a count that leaves these out)
    __builtin_amdgcn_s_barrier();
    read_b(c0{}, bc);
    read_a(0, 0, av[0]);
    lgkm_wait<RB>(bc);
    scale_bias(0);
#pragma unroll
    for (int t = 0; t < NB; ++t) {
        bfr[0][t] = deq_word(bc[t].x, sf[t], bf[t]);
    }
    auto mma = [&](int cur) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            const bf16x8_t af = __builtin_bit_cast(bf16x8_t, av[cur][rb]);
#pragma unroll
            for (int mat = 0; mat < NMAT; ++mat)
#pragma unroll
                for (int cb = 0; cb < NBW; ++cb)
                    acc[mat][rb][cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[cur][mat * NBW + cb], af,
                                                                               acc[mat][rb][cb], 0, 0, 0);
        }
    };
    // Stage u of scale block j (LAST: the last one).  On entry the stage's
    // codes are in registers, its A is published and step 0's fragments are
    // underway.
    auto stage = [&](uint32_t j, auto u_c, auto last_c) {
        constexpr int u = decltype(u_c)::value;
        constexpr bool LAST = decltype(last_c)::value;
        constexpr bool NEXT = !LAST || u + 1 < 8;       // stage s + 1 exists
        constexpr bool MOREA = !LAST || u + NSA < 8;    // stage s + NSA exists
        const uint32_t s = 8u * j + u;
        // the second half of this code block is in registers: refill its slot
        constexpr bool REFILL = (u & 1) != 0 && (!LAST || u < 4);
        if constexpr (REFILL) {
            issue_b(4u * j + (u - 1) / 2 + 2u, std::integral_constant<int, ((u - 1) / 2) & 1>{});
        }
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const int cur = t & 1, nxt = cur ^ 1;
            read_a(s, t + 1, av[nxt]);
            lgkm_wait<RB>(av[cur]);
            // (written ahead of this step's MFMAs it is spread over more of them:
            // 4095 x 11776 x 2048 181 -> 177 us)
#pragma unroll
            for (int f = 0; f < NB; ++f) {
                bfr[nxt][f] = deq_word(word(bc[f], t + 1), sf[f], bf[f]);
            }
            mma(cur);
        }
        // Before the last step: the wave's reads of this A slot are done and
        // its loads of stage s + 1 have landed; the barrier publishes stage
        // s + 1 and frees the slot.
        lgkm_wait<0>(av[1]);
        if constexpr (NEXT) {
            // issued after A(s + 1): A(s + 2), and the last
            // refill (of this stage if odd, of the one before if even)
            constexpr bool REFILL1 = (u & 1) == 0 && (u == 0 || !LAST || u - 1 < 4);
            constexpr bool A2 = !LAST || u + 2 < 8;
            wait_vmcnt<(A2 ? QA : 0) + (REFILL || REFILL1 ? 2 * NB : 0)>();
            __builtin_amdgcn_s_barrier();
            if constexpr (MOREA) {
                issue_a(s + NSA);
            }
            read_b(std::integral_constant<int, (u + 1) & 7>{}, bc);
            read_a(s + 1u, 0, av[0]);
        }
        mma(1);
        if constexpr (NEXT) {
            lgkm_wait<RB>(bc);
            if constexpr (u == 7) {
                if ((j + 1u) % kThinJ == 0u) {
                    load_sb(j + 1u);
                } else {
#pragma unroll
                    for (int t = 0; t < NB; ++t)
#pragma unroll
                        for (int i = 0; i + 1 < kThinJ; ++i) sbr[t][i] = sbr[t][i + 1];
                }
            }
            scale_bias((u + 1) & 7);
#pragma unroll
            for (int f = 0; f < NB; ++f) {
                bfr[0][f] = deq_word(bc[f].x, sf[f], bf[f]);
            }
        }
    };
    for (uint32_t j = 0; j + 1u < nj; ++j) {
        static_for<8>([&](auto u) { stage(j, u, std::false_type{}); });
    }
    static_for<8>([&](auto u) { stage(nj - 1u, u, std::true_type{}); });
    // every wave is done with the LDS before another pass refills it
    __builtin_amdgcn_s_barrier();
    seg_store<RB, NBW, NMAT, EPI>(a, acc, n0, mp0, m_end, i32, h, wave);
}

// An entry of a launch-ordered map (up to 512 rows of one expert) is covered
// in balanced passes of at most RBMAX row blocks, dealt out to `parts`
// workgroups: pass p to workgroup p % parts.  All of an entry's passes read
// the same codes, so its workgroups run on one XCD and near each other; but
// parts without a pass end at once, and runs of them as short as an entry's
// column tiles would leave the live ones on the same few CUs (workgroups are
// dealt to an XCD's 32 CUs in turn), hence the groups of 32 tiles or more.
template <int RBMAX, int NBW, int NMAT, bool GATHER, int EPI>
__global__ __launch_bounds__(kThinWaves * 64, (ThinLayout<RBMAX, NMAT * NBW>::WGS)) void k_thin(GemmArgs a) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lds0 = static_cast<uint32_t>((uintptr_t)((lds_ptr)lds));
    uint4 blk;
    uint32_t part = 0u, parts = 1u;
    if (a.blocks == nullptr) {  // dense: row tiles of dense_bm, fastest, by column tiles
        const uint32_t rt = (a.s_rows + a.dense_bm - 1u) / a.dense_bm;
        const uint32_t mr = (blockIdx.x % rt) * a.dense_bm, nc = (blockIdx.x / rt) * (kThinWaves * NBW * 32u);
        blk = make_uint4(mr, nc, nc, min(mr + a.dense_bm, a.s_rows));
    } else {
        // groups of part_units map rows (their nt column tiles each): part 0
        // of the group's entries, then part 1, ...
        parts = a.parts;
        const uint32_t nt = a.n / (kThinWaves * NBW * 32u), j = blockIdx.x / 8u;
        const uint32_t units = gridDim.x / (8u * parts * nt), per = a.part_units * nt;
        const uint32_t g = j / (per * parts), r = j % (per * parts);
        const uint32_t size = min(a.part_units, units - g * a.part_units) * nt;
        part = r / size;
        blk = a.blocks[(g * per + r % size) * 8u + blockIdx.x % 8u];
    }
    const uint32_t m0 = blk.x, m_end = blk.w;
    if (m0 >= m_end) {
        return;
    }
    const uint32_t nrb = (m_end - m0 + 31u) / 32u;
    const uint32_t passes = (nrb + RBMAX - 1u) / RBMAX;
    const uint32_t each = nrb / passes, extra = nrb % passes;
    for (uint32_t p = part; p < passes; p += parts) {
        const uint32_t mp0 = m0 + 32u * (p * each + min(p, extra));
        const uint32_t rb = each + (p < extra ? 1u : 0u);
        static_for<RBMAX>([&](auto i) {
            if (rb == i + 1u) {
                thin_pass<i + 1, RBMAX, NBW, NMAT, GATHER, EPI>(a, blk.y, blk.z, mp0, m_end, lds0, lane, wave);
            }
        });
    }
}

template <int RBMAX, int NBW, int NMAT, bool GATHER, int EPI>
int launch_thin(const GemmArgs& a, uint32_t n_entries, hipStream_t s) {
    constexpr int lds = ThinLayout<RBMAX, NMAT * NBW>::LDS;
    auto kern = k_thin<RBMAX, NBW, NMAT, GATHER, EPI>;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
        return hip_error(e, "k_thin");
    }
    hipLaunchKernelGGL(kern, dim3(a.blocks == nullptr ? n_entries : n_entries * a.parts), dim3(kThinWaves * 64), lds, s, a);
    return launch_status("k_thin");
}

template <int RBMAX, int NBW>
int launch_dense(GemmArgs g, hipStream_t s) {
    g.dense_bm = 32u * RBMAX;
    const uint32_t tiles = (g.s_rows + g.dense_bm - 1u) / g.dense_bm * (g.n / (kThinWaves * NBW * 32u));
    return launch_thin<RBMAX, NBW, 1, false, EPI_STORE>(g, tiles, s);
}

}  // namespace

namespace mh {

// Whether these kernels run a launch-ordered product (its offset and
// alignment limits checked as the segment kernel's): scales and biases are
// read 16 bytes at a time (make_args leaves the second matrix's null where
// there is one).  The segment kernel covers an expert of up to 288 rows in
// one pass and dequantizes its codes once: a few percent at best.  Steps with
// 208 to 288 rows per expert in the mean, us on the segment kernel against
// these: routed evenly, 64 experts of 2048 x 1536, 4096 tokens 368 to 393 / 378
// to 390 in single passes (on three cards of four 2.5 to 4% slower here), 401 to
// 412 / 388 to 389 with the clocks of a long run; 128 experts 802 / 792, 48
// experts 331 / 302 (2.25 rounds of its workgroups); unevenly (a selection
// bias), 64 experts 440 / 393, 128 experts 892 / 798, 256 experts of 1024 x 512
// 519 / 468.  The host knows only the mean.
bool thin_fits(const GemmArgs& a) {
    return a.ordered && a.stamps == nullptr && aligned(a.s0, 16) && aligned(a.b0, 16) && aligned(a.s1, 16) &&
           aligned(a.b1, 16);
}

template <int NBW, int NMAT, bool GATHER, int EPI>
static int launch_grouped(GemmArgs g, uint32_t n_entries, uint32_t n_experts, hipStream_t s) {
    // One row block per pass needs less LDS (three workgroups per CU): up to a
    // mean of 4 rows (step of 64 experts of 2048 x 1536 top-4, 64 tokens 97 us
    // against 102; 256 experts of 2048 x 512, 255 tokens 118 / 129).  An expert
    // that many tokens choose takes several passes then, dealt out to
    // up to four workgroups: 64 experts top-2, 128 tokens, one expert chosen by
    // all 149 -> 96 us, 256 experts top-4, 255 tokens 228 -> 152.  The first parts of all entries are
    // launched before the others, most of which have no pass: in groups as
    // below those take places among the live ones (64 tokens, no such expert,
    // 97 us with one part, 98 so, 105 in groups).
    const uint32_t nt = g.n / (kThinWaves * NBW * 32u);
    if (g.s_rows <= 4u * n_experts) {
        g.parts = std::min(4u, (g.expert_rows + 31u) / 32u);
        g.part_units = n_entries / (8u * nt);
        return launch_thin<1, NBW, NMAT, GATHER, EPI>(g, n_entries, s);
    }
    g.part_units = (32u + nt - 1u) / nt;
    // a workgroup for every pass of a 512-row entry (step of 255, 1023, 2048,
    // 4096 tokens: 133 178 242 392 us; one workgroup per entry 135 187 266
    // 422, the segment kernel 185 213 285 408)
    g.parts = 4u;
    return launch_thin<4, NBW, NMAT, GATHER, EPI>(g, n_entries, s);
}

int gemm_gu_act_thin(const GemmArgs& a, uint32_t n_entries, hipStream_t s) {
    return launch_grouped<1, 2, true, EPI_SWIGLU>(a, n_entries, a.w_rows / a.n, s);
}

int gemm_grouped_thin(const GemmArgs& a, uint32_t n_entries, hipStream_t s) {
    return launch_grouped<2, 1, false, EPI_STORE>(a, n_entries, a.w_rows / a.n, s);
}

// The dense product: the smallest tile that keeps one workgroup per CU, then
// the widest (rows x columns of 64 x 128, 128 x 128, 128 x 256; us at K 2048,
// one card, in a graph): 255 x 6144 15.7 20.2 27.2; 1023 x 2048 16.1 19.3 27.4;
// 400 x 6144 23.3 21.1 29.0; 1023 x 6144 38.7 36.5 35.3; 2047 x 6144 71.6 61.4
// 61.5; 4095 x 2048 50.3 42.3 40.9; 4095 x 6144 141 120 108; 4095 x 11776 263
// 230 205.  At K 11776: 1023 x 2048 82.9 96.8 140; 2047 x 2048 139 121 150.
int gemm_dense_thin(const GemmArgs& a, hipStream_t s) {
    auto tiles = [&](uint32_t rows) { return (a.s_rows + rows - 1u) / rows * static_cast<uint64_t>(a.n / 128u); };
    if (tiles(64u) <= 256u) {
        return launch_dense<2, 1>(a, s);
    }
    if (tiles(128u) <= 768u || a.n % 256u != 0u) {
        return launch_dense<4, 1>(a, s);
    }
    return launch_dense<4, 2>(a, s);
}

}  // namespace mh
