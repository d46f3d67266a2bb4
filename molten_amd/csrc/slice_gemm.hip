// slice_gemm.hip -- the dense Q4 product of a prefill projection with few
// output tiles (short prompts, narrow matrices): C = A . W^T.
//
// With tiles of 128 x 256 a 255 x 2048 x 2048 product gives 16 workgroups,
// each a serial chain over the whole K: 58 us for 2.1 GFLOP.  Here a tile is
// 32 RB rows x 32 columns and its K is cut into KS slices, one per wave of
// the workgroup, so that the product fills the chip (256 workgroups of 8
// waves) and a wave's chain is 256 k: 7.4 us, half of it the launch and the
// first loads.  What bounds it then is A, which every 32 columns read again
// from the L2 (64 MB here, about 15 TB/s); from a few hundred workgroups on
// thin_gemm.hip's wider tiles are the better ones.
#include "mh_device.hpp"
#include "mh_host.hpp"
#include "mh_q4gemm.hpp"

namespace {

using namespace mh;

struct SliceArgs {
    const uint16_t* a;  // [m, k]
    const uint32_t* codes;
    const uint16_t* scales;
    const uint16_t* biases;
    uint16_t* c;        // [m, n]
    uint32_t m, n, k, row_tiles;
};

// A wave's LDS: two slots, each one stage of 64 k (A rows, codes, scale and
// bias words); after the loop the wave's partial tile.
template <int RB, int KS>
struct SliceLayout {
    static constexpr int A = RB * 4096;
    static constexpr int SLOT = A + 1024 + 256;
    static constexpr int WAVE = 2 * SLOT;
    static constexpr int LDS = KS * WAVE;
    static constexpr int OPS = RB * 4 + 2;  // loads per stage
    static_assert(LDS <= 160 * 1024, "LDS per workgroup");
};

// Wave w takes the 128-k blocks [w nb / KS, (w + 1) nb / KS) of its tile:
// nothing is shared between waves before the sum, so there is no barrier in
// the loop; a slot is read into registers whole and refilled at once.
template <int RB, int KS>
__global__ __launch_bounds__(KS * 64, 1) void k_slice(SliceArgs a) {
    using L = SliceLayout<RB, KS>;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    // all row tiles of a column block on one XCD (its codes stay in that L2)
    const uint32_t j = blockIdx.x / 8u;
    const uint32_t col0 = ((j / a.row_tiles) * 8u + blockIdx.x % 8u) * 32u;
    const uint32_t row0 = (j % a.row_tiles) * (32u * RB);
    if (col0 >= a.n) {
        return;
    }
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i32 = lane & 31, h = lane >> 5;
    const uint32_t K = a.k, nb = K / 128u;
    const uint32_t g0 = 2u * (static_cast<uint32_t>(wave) * nb / KS);
    const uint32_t ng = 2u * ((static_cast<uint32_t>(wave) + 1u) * nb / KS) - g0;  // stages
    const uint32_t own = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>((uintptr_t)((lds_ptr)lds)) + wave * L::WAVE);

    const gbytes abase = uniform_ptr(a.a), cbase = uniform_ptr(a.codes);
    // A load q: rows 8q .. 8q + 7, 128 bytes each; chunk c of row r at c ^ ((r >> 1) & 7)
    uint32_t aoffs[RB * 4];
#pragma unroll
    for (int q = 0; q < RB * 4; ++q) {
        const uint32_t r = 8u * q + static_cast<uint32_t>(lane >> 3);
        const uint32_t chunk = static_cast<uint32_t>(lane & 7) ^ ((r >> 1) & 7u);
        aoffs[q] = min(row0 + r, a.m - 1u) * K * 2u + chunk * 16u + g0 * 128u;
    }
    // codes: 32 bytes per column, chunk c of column i at c ^ ((i >> 3) & 1)
    const uint32_t bcol = static_cast<uint32_t>(lane) >> 1;
    const uint32_t boff = (col0 + bcol) * (K / 2u) + ((static_cast<uint32_t>(lane) ^ (bcol >> 3)) & 1u) * 16u + g0 * 32u;
    // scale (lanes 0-31) and bias (32-63) words: two groups each
    const gbytes sbsrc = (h ? uniform_ptr(a.biases) : uniform_ptr(a.scales)) +
                         ((col0 + static_cast<uint32_t>(i32)) * (K / 64u) + g0) * 2u;
    auto issue = [&](uint32_t s) {
        const uint32_t buf = __builtin_amdgcn_readfirstlane(own + (s & 1u) * L::SLOT);
        const gbytes ag = uniform_ptr(abase + s * 128u);
        static_for<RB * 4>([&](auto q) { dma16m<q * 1024>(ag, aoffs[q], buf); });
        dma16m<L::A>(uniform_ptr(cbase + s * 32u), boff, buf);
        dma4v<L::A + 1024>(sbsrc + (s & ~1u) * 2u, buf);
    };
    f32x16_t acc[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[rb][q] = 0.0f;
    const uint32_t aat = static_cast<uint32_t>(i32) * 128u;
    const uint32_t asw = (static_cast<uint32_t>(i32) >> 1) & 7u;
    const uint32_t bat = L::A + static_cast<uint32_t>(i32) * 32u + ((static_cast<uint32_t>(h) ^ (static_cast<uint32_t>(i32) >> 3)) & 1u) * 16u;
    if (ng > 0u) {
        issue(0);
        issue(1);  // (ng is even)
    }
    for (uint32_t s = 0; s < ng; ++s) {
        if (s + 1u < ng) {
            wait_vmcnt<L::OPS>();
        } else {
            wait_vmcnt<0>();
        }
        const uint32_t buf = own + (s & 1u) * L::SLOT;
        uint4 bc[1], av[4 * RB];
        uint32_t sbw[2];
        bc[0] = lds_read16(buf + bat);
        sbw[0] = lds_read4_at<L::A + 1024>(buf + i32 * 4u);
        sbw[1] = lds_read4_at<L::A + 1024 + 128>(buf + i32 * 4u);
        static_for<4>([&](auto t) {
            const uint32_t at = buf + aat + ((static_cast<uint32_t>(4 * h + t) ^ asw) * 16u);
            static_for<RB>([&](auto rb) { av[t * RB + rb] = lds_read16_at<rb * 4096>(at); });
        });
        lgkm_wait<0>(av);
        lgkm_wait<0>(bc);
        lgkm_wait<0>(sbw);
        if (s + 2u < ng) {
            issue(s + 2u);
        }
        const uint32_t up = (s & 1u) ? 0u : 16u;  // an odd group's bf16 is the word's high half
        const float sf = __uint_as_float((sbw[0] << up) & 0xffff0000u);
        const float bf = __uint_as_float((sbw[1] << up) & 0xffff0000u);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint32_t wv = t == 0 ? bc[0].x : t == 1 ? bc[0].y : t == 2 ? bc[0].z : bc[0].w;
            const bf16x8_t w = deq_word(wv, sf, bf);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                acc[rb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, __builtin_bit_cast(bf16x8_t, av[t * RB + rb]),
                                                                  acc[rb], 0, 0, 0);
            }
        }
    }
    // The partial tile (row 32 rb + i32, columns 8p + 4h .. + 3 at q = 4p) into
    // the wave's own LDS: 16-byte piece c of row r at c ^ (r & 7).
    float* part = reinterpret_cast<float*>(lds + wave * L::WAVE);
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const uint32_t r = 32u * rb + static_cast<uint32_t>(i32);
            const uint32_t at = r * 8u + ((static_cast<uint32_t>(2 * p + h)) ^ (r & 7u));
            *reinterpret_cast<float4*>(part + 4u * at) =
                make_float4(acc[rb][4 * p], acc[rb][4 * p + 1], acc[rb][4 * p + 2], acc[rb][4 * p + 3]);
        }
    __syncthreads();
    // the slices' sum, in slice order, four columns per thread
    for (uint32_t i = threadIdx.x; i < 32u * RB * 8u; i += KS * 64u) {
        const uint32_t r = i >> 3, c = i & 7u;
        if (row0 + r >= a.m) {
            break;  // later pieces are of later rows
        }
        const uint32_t at = 4u * (r * 8u + (c ^ (r & 7u)));
        float4 v = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(lds) + at);
#pragma unroll
        for (int w = 1; w < KS; ++w) {
            const float4 u = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(lds + w * L::WAVE) + at);
            v.x += u.x; v.y += u.y; v.z += u.z; v.w += u.w;
        }
        const uint2 o = make_uint2(pack_bf16(v.x, v.y), pack_bf16(v.z, v.w));
        *reinterpret_cast<uint2*>(a.c + static_cast<size_t>(row0 + r) * a.n + col0 + 4u * c) = o;
    }
}

template <int RB, int KS>
int launch_slice(SliceArgs a, hipStream_t s) {
    constexpr int lds = SliceLayout<RB, KS>::LDS;
    a.row_tiles = (a.m + 32u * RB - 1u) / (32u * RB);
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_slice<RB, KS>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
        return hip_error(e, "k_slice");
    }
    hipLaunchKernelGGL((k_slice<RB, KS>), dim3((a.n / 32u + 7u) / 8u * 8u * a.row_tiles), dim3(KS * 64), lds, s, a);
    return launch_status("k_slice");
}

}  // namespace

namespace mh {

// The smallest tile that keeps one workgroup per CU (us at K 2048 / 11776 by
// tile, in a graph: 32 rows 8 slices, 64 rows 8, 64 rows 4, 128 rows 4; then
// the tiles of thin_gemm.hip): 21 x 2048 rows and columns 5.1 6.4 6.3 8.7, 12.5
// / 14 20 22 30, 59; 255 x 2048 9.8 7.4 7.1 9.6, 14.0 / 50 35 36 45, 72; 500 x
// 2048 17.9 13.0 11.7 10.6, 14.3; 100 x 6144 13.4 11.9 10.5 9.7, 14.6; 60 x
// 11776 13.5 12.3 10.6 16.3, 14.1.  Past that (255 x 6144: 25.7 19.3 16.1 17.6)
// those take 16.0.
//
// The slices are summed apart, 8 or 4 by the tile, so a row's f32 sum runs in
// another order than on the kernels without them: its bits follow m and n.
bool gemm_dense_slices(const uint16_t* a, uint32_t m, const mh_quant_weights* w, uint16_t* c, hipStream_t s, int* rc) {
    const uint32_t n = w->out_features, k = w->in_features;
    // 128-k blocks, 32-bit byte offsets, 8-byte stores and whole code pieces; no
    // tall A, which every column block reads again, from memory past the L2s
    // (16000 rows x 64 columns, K 2048 / 11776: 59 / 340 us against 54 / 266 on
    // 128-row tiles, 12000 45 / 250 against 54 / 266)
    if (k % 128u != 0u || n % 32u != 0u || m > 12288u || !aligned(c, 8) || !aligned(w->codes, 16) ||
        !aligned(w->scales, 4) || !aligned(w->biases, 4) || static_cast<uint64_t>(m) * k * 2u >= (1ull << 32) ||
        static_cast<uint64_t>(n) * k / 2u >= (1ull << 32)) {
        return false;
    }
    const SliceArgs g{a, w->codes, w->scales, w->biases, c, m, n, k, 0u};
    const uint64_t cb = n / 32u;
    auto tiles = [&](uint32_t rows) { return (m + rows - 1u) / rows * cb; };
    if (m <= 32u || tiles(32u) <= 256u) {
        *rc = launch_slice<1, 8>(g, s);
    } else if (tiles(64u) <= 256u) {
        *rc = launch_slice<2, 8>(g, s);
    } else if (tiles(128u) <= 256u) {
        *rc = launch_slice<4, 4>(g, s);
    } else if (tiles(64u) <= 512u) {
        *rc = launch_slice<2, 4>(g, s);
    } else {
        return false;
    }
    return true;
}

}  // namespace mh
