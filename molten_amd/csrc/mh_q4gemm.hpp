// mh_q4gemm.hpp -- what the Q4 matrix-product kernels share (grouped_gemm.hip,
// thin_gemm.hip): their argument block, the dequantization of a code word
// into an MFMA fragment, and the epilogue that stores a wave's tiles.
#pragma once

#include <type_traits>

#include "mh_mfma.hpp"

namespace mh {

constexpr int kBK = 64;

enum Epi { EPI_STORE = 0, EPI_GATE_UP = 1, EPI_SWIGLU = 2 };

struct GemmArgs {
    const uint16_t* a;       // [a_rows, k] bf16
    const uint32_t* gather;  // row i of the tile reads a[gather[i]]; null: a[i]
    const uint32_t* c0; const uint16_t* s0; const uint16_t* b0;  // gate / the matrix
    const uint32_t* c1; const uint16_t* s1; const uint16_t* b1;  // up
    uint16_t* out0;          // [s_rows, n]: C, gate, or act
    uint16_t* out1;          // [s_rows, n]: up (EPI_GATE_UP)
    const uint4* blocks;     // block map; null: a dense product (entries computed)
    uint32_t k, n, s_rows, a_rows, w_rows;
    uint32_t expert_rows;    // k_thin: rows an expert is taken to have at most (sizes its parts)
    uint32_t dense_bm;       // rows per entry of a dense product
    uint32_t parts;          // k_thin: workgroups per map entry (its passes dealt out in turn)
    uint32_t part_units;     // k_thin: map rows whose parts are launched part by part
    uint32_t ordered;        // k_seg: the map is in launch order (entry b for workgroup b)
    uint64_t* stamps;        // per workgroup MH_PREFILL_STAMPS words (stamped k_seg only), or null
};

// thin_gemm.hip: launch-ordered products.
bool thin_fits(const GemmArgs& a);
int gemm_gu_act_thin(const GemmArgs& a, uint32_t n_entries, hipStream_t s);
int gemm_grouped_thin(const GemmArgs& a, uint32_t n_entries, hipStream_t s);
// thin_gemm.hip: the dense product (n % 128 == 0, k % 512 == 0, the segment
// kernel's offset and alignment limits).
int gemm_dense_thin(const GemmArgs& a, hipStream_t s);
// slice_gemm.hip: the dense product with few output tiles; false where its
// shape, size or alignment is not taken.
bool gemm_dense_slices(const uint16_t* a, uint32_t m, const mh_quant_weights* w, uint16_t* c, hipStream_t s, int* rc);

// One Q4 word (8 codes, low nibble first) -> bf16(fma(s, q, b)) x 8.  A code
// in a byte of its own is the fp8 (e4m3) denormal q 2^-9, so one scaled
// conversion gives two codes as f32 q exactly, whatever s: 19 VALU
// instructions a word instead of the 22 with one v_cvt_f32_ubyte a code (54
// against 68 cycles of a SIMD shared by two waves: conversions and bf16 packs
// take 4, fma and logic 2).  Prefill step of 255 tokens 192.6 -> 184.1 us,
// projection 4095 x 6144 x 2048 114.1 -> 112.0 us; the 4096-token step, whose
// MFMAs hide the dequant, 369 us either way.
__device__ __forceinline__ bf16x8_t deq_word(uint32_t w, float s, float b) {
    const uint32_t lo = opaque(w & 0x0f0f0f0fu);
    const uint32_t hi = opaque((w >> 4) & 0x0f0f0f0fu);
    uint32_t p[4];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const f32x2_t e = j == 0 ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(static_cast<int>(lo), 512.0f, false)
                                 : __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(static_cast<int>(lo), 512.0f, true);
        const f32x2_t o = j == 0 ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(static_cast<int>(hi), 512.0f, false)
                                 : __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(static_cast<int>(hi), 512.0f, true);
        p[2 * j] = pack_bf16(__builtin_fmaf(e[0], s, b), __builtin_fmaf(o[0], s, b));
        p[2 * j + 1] = pack_bf16(__builtin_fmaf(e[1], s, b), __builtin_fmaf(o[1], s, b));
    }
    const uint4 u = make_uint4(p[0], p[1], p[2], p[3]);
    return __builtin_bit_cast(bf16x8_t, u);
}

// Compile-time loop: f(std::integral_constant<int, i>) for i in [0, N).
template <int I, int N, typename F>
__device__ __forceinline__ void static_for_impl(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for_impl<I + 1, N>(f);
    }
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl<0, N>(f);
}

// Fast SiLU for the GEMM epilogue (the gate/up values it sees already
// carry MFMA accumulation error): g * 1 / (1 + 2^(-g log2 e)) with the
// hardware exp2 and reciprocal (1 ulp each).
__device__ __forceinline__ float silu_hw(float g) {
    const float e = __builtin_amdgcn_exp2f(g * -1.4426950408889634f);
    return g * __builtin_amdgcn_rcpf(1.0f + e);
}

__device__ __forceinline__ float bf16_round_hw(float v) {
    const f32x2_t p = {v, 0.0f};
    const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector(p, bf16x2_t));
    return __uint_as_float(u << 16);
}

// Epilogue of the kernels whose MFMAs compute C^T: stores the wave's RB row
// blocks of rows mp0 .. m_end - 1 (row block rb, lane i32: row mp0 + 32 rb +
// i32) at columns n0 + 32 (wave NBW + cb) .. + 31.
template <int RB, int NBW, int NMAT, int EPI>
__device__ __forceinline__ void seg_store(const GemmArgs& a, const f32x16_t (&acc)[NMAT][RB][NBW], uint32_t n0,
                                          uint32_t mp0, uint32_t m_end, int i32, int h, int wave) {
    // The MFMAs computed C^T (W fragment as the first
    // operand): lane (i32, h) holds row mp0 + 32 rb + i32 and, at q = 4p + r,
    // column 8p + 4h + r of its 32-column block.  Values become bf16 pairs;
    // permlane32_swap of the (p even, p odd) pairs gives lane h = 0 columns
    // 8p..8p+7 of p = 0, 2 and lane h = 1 those of p = 1, 3, stored 16 bytes
    // at a time.
    const gbytes ob0 = uniform_ptr(reinterpret_cast<const char*>(a.out0));
    const gbytes ob1 = uniform_ptr(reinterpret_cast<const char*>(a.out1 ? a.out1 : a.out0));
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        const uint32_t row = mp0 + rb * 32u + static_cast<uint32_t>(i32);
#pragma unroll
        for (int cb = 0; cb < NBW; ++cb) {
            constexpr int NOUT = (EPI == EPI_GATE_UP) ? 2 : 1;
            uint32_t w[NOUT][4][2];  // [output][p][pair]
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                float v[NOUT][4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int q = 4 * p + r;
                    if constexpr (EPI == EPI_SWIGLU) {
                        const float g = bf16_round_hw(acc[0][rb][cb][q]);
                        const float u = bf16_round_hw(acc[1][rb][cb][q]);
                        v[0][r] = bf16_round_hw(silu_hw(g)) * u;
                    } else {
#pragma unroll
                        for (int o = 0; o < NOUT; ++o) {
                            v[o][r] = acc[o][rb][cb][q];
                        }
                    }
                }
#pragma unroll
                for (int o = 0; o < NOUT; ++o) {
                    w[o][p][0] = pack_bf16(v[o][0], v[o][1]);
                    w[o][p][1] = pack_bf16(v[o][2], v[o][3]);
                }
            }
            const uint32_t col = n0 + static_cast<uint32_t>((wave * NBW + cb) * 32 + 8 * h);
            const uint32_t off = (row * a.n + col) * 2u;
#pragma unroll
            for (int o = 0; o < NOUT; ++o) {
#pragma unroll
                for (int pp = 0; pp < 2; ++pp) {
#pragma unroll
                    for (int d = 0; d < 2; ++d) {
                        const auto r = __builtin_amdgcn_permlane32_swap(w[o][2 * pp][d], w[o][2 * pp + 1][d], false, false);
                        w[o][2 * pp][d] = r[0];
                        w[o][2 * pp + 1][d] = r[1];
                    }
                }
                if (row < m_end) {
                    const gbytes ob = o == 0 ? ob0 : ob1;
                    typedef __attribute__((address_space(1))) u32x4* g4;
                    // columns 8h .. 8h+7 (pp = 0) and 16 + 8h .. (pp = 1)
                    *reinterpret_cast<g4>(const_cast<char __attribute__((address_space(1)))*>(ob) + off) =
                        u32x4{w[o][0][0], w[o][0][1], w[o][1][0], w[o][1][1]};
                    *reinterpret_cast<g4>(const_cast<char __attribute__((address_space(1)))*>(ob) + off + 32u) =
                        u32x4{w[o][2][0], w[o][2][1], w[o][3][0], w[o][3][1]};
                }
            }
        }
    }
}

}  // namespace mh
