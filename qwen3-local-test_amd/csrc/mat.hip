// The projections on either side of the attention layer for gfx950: Y[n][rows] = X[n][cols] W^T with W in
// planar Q8_0 (int8 weights, one f32 scale per 32 consecutive weights of a row) or plain f32 rows.
//
// Replaces Qwen4Vulkan::mat (src/qwen4_vk.cpp:848-856) on its matrix-vector pipelines q4_matmul_q8 /
// q4_matmul_f32 (shaders/q4_matmul.comp with the C_Q8 / C_F32 codecs of shaders/q4_codec.glsl; the planar
// repacking of GGUF Q8_0 is src/qwen4_vk.cpp:98-106) and on its tiled GEMM pipelines q4_gemm_q8 / q4_gemm_f32:
// every output is the fp32 dot product of a dequantized weight row (int8 times its block's scale) with a
// token's input row, then optionally silu(y * post_scale). One token, and fp32 weights below 16: matrix-vector
// kernels. Q8 from two tokens to a few hundred: the token-tile MFMA kernel. Beyond, and fp32 weights from 16:
// the tiled MFMA GEMM.
//
// MI355X design of the matrix-vector kernels: the weights are read once per launch and are the bound (a
// decode step's projections are memory-bound); a wave owns RW rows and a workgroup one token (f32: up to four),
// lane l covering the 16 consecutive columns 16 l + 1,024 k of every row, so a wave reads a kilobyte of each row
// per chunk in one 16-byte load a lane (plus one scale a lane pair), and every weight load of a wave's rows is
// issued before the first is used. A 16-column group never crosses a 32-weight block, so the lane applies its
// block scale once per group. The partial dot products are summed over the wave with DPP row operations and
// permlane swaps.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace qw {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kMatNTP = 4;  // tokens a workgroup (f32 weights)

// Sum over the 64 lanes, in every lane.
__device__ __forceinline__ float mat_wave_sum(float x) {
    x = sum32(x);
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
}

// f32 weights: a wave's RW rows a 16-column group at a time (f32 projections are the small ones)
template <int NTP, int RW>
__device__ __forceinline__ void mat_f32_body(const MatArgs& a, int bx) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int r0 = (bx * 4 + wave) * RW;
    const int t0 = blockIdx.y * NTP;
    const int nt = min(NTP, a.n - t0);
    if (r0 >= a.rows) return;  // whole waves
    float acc[RW][NTP];
#pragma unroll
    for (int r = 0; r < RW; r++)
#pragma unroll
        for (int t = 0; t < NTP; t++) acc[r][t] = 0.f;
    for (int c = lane * 16; c < a.cols; c += 1024) {
        float xv[NTP][16];
#pragma unroll
        for (int t = 0; t < NTP; t++) {
            const float* xr = a.x + (size_t)(t0 + (t < nt ? t : 0)) * a.x_stride + c;
#pragma unroll
            for (int i = 0; i < 16; i += 4) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(xr + i);
                xv[t][i] = v[0], xv[t][i + 1] = v[1], xv[t][i + 2] = v[2], xv[t][i + 3] = v[3];
            }
        }
#pragma unroll
        for (int r = 0; r < RW; r++) {
            const float* wr = static_cast<const float*>(a.w) + (size_t)min(r0 + r, a.rows - 1) * a.cols + c;
            float wv[16];
#pragma unroll
            for (int i = 0; i < 16; i += 4) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(wr + i);
                wv[i] = v[0], wv[i + 1] = v[1], wv[i + 2] = v[2], wv[i + 3] = v[3];
            }
#pragma unroll
            for (int t = 0; t < NTP; t++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc[r][t] = __builtin_fmaf(wv[i], xv[t][i], acc[r][t]);
        }
    }
#pragma unroll
    for (int r = 0; r < RW; r++)
#pragma unroll
        for (int t = 0; t < NTP; t++) {
            float v = mat_wave_sum(acc[r][t]);
            if (a.post == 1) {
                const float u = v * a.post_scale;
                v = u / (1.0f + __expf(-u));
            }
            if (lane == 0 && r0 + r < a.rows && t < nt) a.y[(size_t)(t0 + t) * a.y_stride + r0 + r] = v;
        }
}

// planar Q8: every weight load of a batch of up to kMatK 1,024-column chunks (RW rows x kMatK 16-byte
// loads a lane, with their scales) is issued before any is used, so a wave has its whole share of the
// matrix in flight at once (the stream is the bound: the loads have to overlap); then per chunk the token
// rows' 16 columns (cached: every wave reads them) and the dot products
constexpr int kMatK = 4;
template <int RW>
__device__ __forceinline__ void mat_q8_body(const MatArgs& a, int bx) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int r0 = (bx * 4 + wave) * RW;
    const int t = blockIdx.y;
    if (r0 >= a.rows) return;  // whole waves
    const int8_t* w8 = static_cast<const int8_t*>(a.w);
    const int nsb = a.cols >> 5;  // scales a row
    float acc[RW];
#pragma unroll
    for (int r = 0; r < RW; r++) acc[r] = 0.f;
    for (int cb = 0; cb < a.cols; cb += kMatK * 1024) {
        u32x4 q[RW][kMatK];
        float sc[RW][kMatK];
#pragma unroll
        for (int k = 0; k < kMatK; k++) {
            if (cb + k * 1024 >= a.cols) break;  // the whole chunk lies past the row (wave-uniform)
            const int c = min(cb + k * 1024 + lane * 16, a.cols - 16);  // past the row: a valid group, unused
#pragma unroll
            for (int r = 0; r < RW; r++) {
                const int row = min(r0 + r, a.rows - 1);  // past the last row: a valid row, result not stored
                q[r][k] = *reinterpret_cast<const u32x4*>(w8 + (size_t)row * a.cols + c);
                sc[r][k] = a.s[(size_t)row * nsb + (c >> 5)];
            }
        }
#pragma unroll
        for (int k = 0; k < kMatK; k++) {
            if (cb + k * 1024 >= a.cols) break;
            const int c = cb + k * 1024 + lane * 16;
            if (c >= a.cols) continue;  // this lane's group lies past the row
            float xv[16];
            const float* xr = a.x + (size_t)t * a.x_stride + c;
#pragma unroll
            for (int i = 0; i < 16; i += 4) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(xr + i);
                xv[i] = v[0], xv[i + 1] = v[1], xv[i + 2] = v[2], xv[i + 3] = v[3];
            }
#pragma unroll
            for (int r = 0; r < RW; r++) {
                float wv[16];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int v = (int)q[r][k][j];
                    wv[4 * j] = (float)((v << 24) >> 24);
                    wv[4 * j + 1] = (float)((v << 16) >> 24);
                    wv[4 * j + 2] = (float)((v << 8) >> 24);
                    wv[4 * j + 3] = (float)(v >> 24);
                }
                float d = 0.f;
#pragma unroll
                for (int i = 0; i < 16; i++) d = __builtin_fmaf(wv[i], xv[i], d);
                acc[r] = __builtin_fmaf(d, sc[r][k], acc[r]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < RW; r++) {
        float v = mat_wave_sum(acc[r]);
        if (a.post == 1) {
            const float u = v * a.post_scale;
            v = u / (1.0f + __expf(-u));
        }
        if (lane == 0 && r0 + r < a.rows) a.y[(size_t)t * a.y_stride + r0 + r] = v;
    }
}

template <int RW>
__global__ __launch_bounds__(256) void k_mat_q8(MatArgs a) {
    mat_q8_body<RW>(a, blockIdx.x);
}
template <int NTP, int RW>
__global__ __launch_bounds__(256) void k_mat_f32(MatArgs a) {
    mat_f32_body<NTP, RW>(a, blockIdx.x);
}

// Several matrices on one input in one launch: workgroups [wg_end[i-1], wg_end[i]) run matrix i (a
// wave-uniform choice), so a decode step's query, key and value projections stream as one burst.
template <bool Q8, int NTP, int RW>
__global__ __launch_bounds__(256) void k_mat_multi(MatMultiArgs a) {
    int i = 0;
    while (i + 1 < a.count && (int)blockIdx.x >= a.wg_end[i]) i++;
    const int bx = (int)blockIdx.x - (i ? a.wg_end[i - 1] : 0);
    if constexpr (Q8) mat_q8_body<RW>(a.m[i], bx);
    else mat_f32_body<NTP, RW>(a.m[i], bx);
}

// ---- fp32 weights, many tokens: tiled MFMA GEMM ---------------------------------------------------------
// Replaces the q4_gemm_f32 pipeline (shaders/q4_gemm.comp) that Qwen4Vulkan::mat selects from nine tokens on
// (src/qwen4_vk.cpp:852-853). A workgroup owns a 128-row x BN-token tile of Y, walks the columns one 32-column
// step at a time through two LDS stages, and its four waves each own a 64-row x BN/2-token quarter as
// 4 x BN/32 v_mfma_f32_16x16x32_bf16 tiles (A = weight rows, B = token rows). fp32 accuracy from bf16 products:
// an fp32 value v is split into hi = bf16(v) and lo = bf16(v - hi), which leaves |v - hi - lo| <= 2^-18 |v|; four
// MFMAs a tile (hi.hi, hi.lo, lo.hi, lo.lo) then carry a product to within 2^-17 before the fp32 accumulation.
// The next step's global loads are in flight while the current step's MFMAs run; tiles are assigned so that each
// XCD takes a contiguous range of row tiles (its weights stay in its L2).
constexpr int kGemmBM = 128;  // rows a workgroup

// Byte offset of 16-byte chunk g (k = 8 g .. 8 g + 7) of tile row r in an LDS tile of [rows][32] bf16: the
// chunk index is XORed with (r / 2) % 4, so any 8 consecutive rows' chunk g (an MFMA operand read) and any
// 4 rows' chunk pairs (the loaders' writes) land in 8 distinct 16-byte bank groups (no bank conflicts,
// counted by SQ_LDS_BANK_CONFLICT).
__device__ __forceinline__ int gemm_off(int r, int g) { return r * 64 + ((g ^ ((r >> 1) & 3)) << 4); }

__device__ __forceinline__ void split_bf16(const float (&v)[8], bf16x8& hi, bf16x8& lo) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
        hi[i] = (__bf16)v[i];
        lo[i] = (__bf16)(v[i] - (float)hi[i]);
    }
}

// ---- two to a few hundred tokens, Q8: token-tile MFMA kernel, the columns split over the waves -----------
// A workgroup owns 16 R rows x 16 TT tokens and its waves split the columns: wave w takes the 128-column quads
// w, w + KW, ... (four Q8 blocks each), so that nothing is loaded or converted twice in a workgroup and no
// barrier is needed before the waves' sums meet. Weights are the B operand: an accumulator column is then a
// weight row, its block scale one value a lane.
//
// What bounds it is the rate of the vector-memory pipe and of instruction issue, not HBM. A load costs one cycle
// per 64-byte piece it touches, so an operand loaded straight in the MFMA layout (lane l: row l % 16) costs 64
// cycles a kilobyte; loaded by consecutive lanes it costs 16, and a pass through the wave's own part of the LDS
// (written as loaded, read as operands, spread over the banks by the XORs below: conflicts are 0.4 of its active
// cycles, and waves wait for it 6% of theirs at 77 tokens; in-order within the wave) gives the layout. 9,216 x 2,048 at 4 / 77 tokens, one box: 10.9 / 31.1 us with operand-layout loads,
// 8.5 / 20.7 us through the LDS; the kernels before (fp32 multiply-adds on up to 4 tokens a workgroup; 32-row
// workgroups with operand-layout loads from 16) took 16.0 / 86 us. A vector instruction, the conversions
// included, takes a SIMD 2.0-2.5 ns.
//
// fp32 accuracy from bf16 products: an int8 weight is exact in bf16; NS = 2 splits x into hi + lo (up to 2^-18 of
// |x| left, 2.5e-6 in an output), NS = 3 into three parts of eight bits (nothing left: 1e-7 in an output, the level of
// fp32 sums), for the token counts below 16. bf16 ends at 2^-133, so the last part of an |x| below 2^-109 loses bits:
// rows whose values are all that small keep 1.2e-6 at 2^-115 and 4e-5 at 2^-120 of their outputs, with two parts
// 2.8e-6 and 4e-5.
__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {  // one v_cvt_pk_bf16_f32
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

// What the bf16 pair w = pk_bf16(v0, v1) leaves of v0 (E = 0) or v1 (E = 1), exactly, in one v_dot2_f32_bf16 with
// (-1, 0) or (0, -1) (an infinity in either makes both NaN). The pair is made opaque: as a constant the compiler
// writes the first as the inline operand -1.0, which the instruction reads as the second.
template <int E>
__device__ __forceinline__ float rest_bf16(uint32_t w, float v) {
    uint32_t m;
    if constexpr (E == 0) asm("s_mov_b32 %0, 0xbf80" : "=s"(m));
    else asm("s_mov_b32 %0, 0xbf800000" : "=s"(m));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w), __builtin_bit_cast(bf16x2, m), v, false);
}

// Eight int8 weights (two words) as bf16, exactly.
__device__ __forceinline__ bf16x8 weights_bf16(uint32_t lo, uint32_t hi) {
    u32x4 w;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int v = (int)(e < 2 ? lo : hi), s = 16 * (e & 1);
        w[e] = pk_bf16((float)((v << (24 - s)) >> 24), (float)((v << (16 - s)) >> 24));
    }
    return __builtin_bit_cast(bf16x8, w);
}

// KW waves; B > 1 (TT = 1, up to 16 / B tokens): B consecutive blocks share the rows of one A operand, block j
// of them in rows [16 j / B, 16 (j + 1) / B), so that their token values are split in one go; a block's product
// is then valid in the lanes of its rows only, which take it with their own block's scale.
template <int TT, int R, int NS, int B>
struct TokLds {  // a wave's part of the LDS
    unsigned char w[R][2048];       // a quad of 16 rows: [row][8 chunks of 16 columns], chunk ^ (row / 2) % 8
    float s[R][64];                 // their scales [row][block]
    unsigned char x[TT][NS][1024];  // an A operand's parts: [8-column group][row ^ 4 group], 16 bytes
};

template <int TT, int R, int NS, int B, int KW>
__device__ __forceinline__ void mat_tok_body(const MatArgs& a, int bx, int by, unsigned char* smem) {
    static_assert(B == 1 || TT == 1, "shared rows: one token tile");
    typedef TokLds<TT, R, NS, B> Lds;
    constexpr int U = 4 / B;                        // A operands a quad
    constexpr int XR = U == 4 && TT >= 3 ? 2 : U;   // token-row buffers: A operands in flight
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int c = lane & 15, g = lane >> 4;
    const int r0 = bx * 16 * R, t0 = by * 16 * TT;
    const int nkb = a.cols >> 5, nq = (nkb + 3) >> 2;
    constexpr size_t kLds = sizeof(Lds) > R * TT * 1024 ? sizeof(Lds) : R * TT * 1024;  // (the final sums reuse it)
    Lds& L = *reinterpret_cast<Lds*>(smem + wave * kLds);
    // rows past the matrix, tokens past the last and columns past the row (kFar added) lie outside the
    // resources: such loads read zero and cause no traffic, so no load is conditional
    const int nr = min(16 * R, a.rows - r0), nt = min(16 * TT, a.n - t0);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(static_cast<const int8_t*>(a.w)) + (size_t)r0 * a.cols, (short)0, nr * a.cols, 0x00020000);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(a.s) + (size_t)r0 * nkb, (short)0, nr * nkb * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(a.x) + (size_t)t0 * a.x_stride, (short)0, ((nt - 1) * a.x_stride + a.cols) * 4, 0x00020000);

    // loads: 16 bytes a lane, whole cache lines by consecutive lanes. Weights: load i of a quad is rows
    // 8 i + lane / 8, chunk lane % 8. Scales: row lane / 4, block lane % 4. Token rows: load i of an A operand is
    // piece 64 i + lane of its [16 / B tokens][32 B columns].
    u32x4 wq[R][2];
    float sq[R];
    f32x4 xv[XR][TT][2];
    auto load_w = [&](int q) {
        const int col = 128 * q + 16 * (lane & 7), blk = 4 * q + (lane & 3);
        const unsigned cw = col < a.cols ? (unsigned)col : kFar, cs = blk < nkb ? 4u * blk : kFar;
#pragma unroll
        for (int r = 0; r < R; r++) {
#pragma unroll
            for (int i = 0; i < 2; i++)
                wq[r][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                    rw, (int)((16 * r + 8 * i + (lane >> 3)) * a.cols + cw), 0, 0));
            sq[r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, (int)((16 * r + (lane >> 2)) * nkb * 4 + cs), 0, 0));
        }
    };
    int xoff[TT][2];  // the pieces' token rows
#pragma unroll
    for (int t = 0; t < TT; t++)
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int p = 64 * i + lane, tok = 16 * t + p / (8 * B);
            xoff[t][i] = tok < nt ? (tok * a.x_stride + 4 * (p % (8 * B))) * 4 : (int)kFar;
        }
    const int xblk = (lane % (8 * B)) / 8;  // this lane's block of the A operand
    auto load_x = [&](auto k_, int b) {
        constexpr int k = k_;
        const unsigned o = b + xblk < nkb ? 128u * b : kFar;
#pragma unroll
        for (int t = 0; t < TT; t++)
#pragma unroll
            for (int i = 0; i < 2; i++)
                xv[k][t][i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, (int)(xoff[t][i] + o), 0, 0));
    };
    // LDS places: of this lane's pieces (written) and fragments (read)
    int wst[2], xst[2], wld[4];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int row = 8 * i + (lane >> 3);
        wst[i] = row * 128 + (((lane & 7) ^ ((row >> 1) & 7)) << 4);
        const int p = 64 * i + lane, xr = (p % (8 * B)) / 8 * (16 / B) + p / (8 * B), pc = p % 8;
        xst[i] = ((pc >> 1) * 16 + (xr ^ ((pc >> 1) << 2))) * 16 + (pc & 1) * 8;
    }
#pragma unroll
    for (int j = 0; j < 4; j++) wld[j] = c * 128 + (((2 * j + (g >> 1)) ^ ((c >> 1) & 7)) << 4) + (g & 1) * 8;
    const int xld = (g * 16 + (c ^ (g << 2))) * 16;

    f32x4 acc[R][TT];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int t = 0; t < TT; t++) acc[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    // first block of the j-th A operand from quad q on
    auto block_of = [&](int q, int j) { return 4 * (q + KW * (j / U)) + B * (j % U); };
    load_w(wave);
    static_for<0, XR>([&](auto j) { load_x(j, block_of(wave, j)); });
#pragma unroll 1
    for (int q = wave; q < nq; q += KW) {
#pragma unroll
        for (int r = 0; r < R; r++) {
#pragma unroll
            for (int i = 0; i < 2; i++) *reinterpret_cast<u32x4*>(L.w[r] + wst[i]) = wq[r][i];
            L.s[r][lane] = sq[r];
        }
        load_w(q + KW);
        float sc[R][U];
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int u = 0; u < U; u++) sc[r][u] = L.s[r][4 * c + (B == 1 ? u : B == 2 ? 2 * u + (g >> 1) : g)];
        static_for<0, U>([&](auto u_) {
            constexpr int u = u_, xb = u % XR;
            // the A operand's token values: split and laid out
#pragma unroll
            for (int t = 0; t < TT; t++)
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    uint32_t part[NS][2];
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        float v0 = xv[xb][t][i][2 * e], v1 = xv[xb][t][i][2 * e + 1];
#pragma unroll
                        for (int k = 0; k < NS; k++) {
                            if (NS == 3 && k == 0) {
                                // three parts: the first cut off, not rounded (which takes the largest finite values
                                // to infinity); an infinity is its first part, as fp32 products would have it
                                const uint32_t b0 = __float_as_uint(v0), b1 = __float_as_uint(v1);
                                part[k][e] = __builtin_amdgcn_perm(b1, b0, 0x07060302u);
                                v0 = __builtin_fabsf(v0) == __builtin_inff() ? 0.f : v0 - __uint_as_float(b0 & 0xFFFF0000u);
                                v1 = __builtin_fabsf(v1) == __builtin_inff() ? 0.f : v1 - __uint_as_float(b1 & 0xFFFF0000u);
                                continue;
                            }
                            const uint32_t w = pk_bf16(v0, v1);
                            part[k][e] = w;
                            if (k + 1 < NS) v0 = rest_bf16<0>(w, v0), v1 = rest_bf16<1>(w, v1);
                        }
                    }
#pragma unroll
                    for (int k = 0; k < NS; k++)
                        *reinterpret_cast<u32x2*>(L.x[t][k] + xst[i]) = u32x2{part[k][0], part[k][1]};
                }
            load_x(std::integral_constant<int, xb>{}, block_of(q, u + XR));
            if (block_of(q, u) < nkb) {  // uniform; a group's blocks past the row hold zeros
                f32x4 p[R][TT];
#pragma unroll
                for (int jj = 0; jj < B; jj++) {
                    bf16x8 wv[R];
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        const u32x2 w = *reinterpret_cast<const u32x2*>(L.w[r] + wld[u * B + jj]);
                        wv[r] = weights_bf16(w[0], w[1]);
                    }
#pragma unroll
                    for (int t = 0; t < TT; t++) {
                        f32x4 d[R];
#pragma unroll
                        for (int i = 0; i < NS; i++) {
                            // (three parts from the last: the first two of a value near the largest may sum to 2^128)
                            const int k = NS == 3 ? NS - 1 - i : i;
                            const bf16x8 part = *reinterpret_cast<const bf16x8*>(L.x[t][k] + xld);
#pragma unroll
                            for (int r = 0; r < R; r++)
                                d[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(part, wv[r], i ? d[r] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                        }
#pragma unroll
                        for (int r = 0; r < R; r++) {
                            if (jj == 0) p[r][t] = d[r];
                            else
#pragma unroll
                                for (int i = 0; i < 4; i++) p[r][t][i] = (g * B) / 4 == jj ? d[r][i] : p[r][t][i];
                        }
                    }
                }
#pragma unroll
                for (int t = 0; t < TT; t++)
#pragma unroll
                    for (int r = 0; r < R; r++)
#pragma unroll
                        for (int i = 0; i < 4; i++) acc[r][t][i] = __builtin_fmaf(sc[r][u], p[r][t][i], acc[r][t][i]);
            }
        });
    }
    // shared rows: the groups of lanes hold the sums of different blocks
    if constexpr (B > 1) {
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                uint32_t v = __float_as_uint(acc[r][0][i]);
                const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);
                float f = __uint_as_float(h[0]) + __uint_as_float(h[1]);
                if constexpr (B == 4) {
                    v = __float_as_uint(f);
                    const auto l = __builtin_amdgcn_permlane16_swap(v, v, false, false);
                    f = __uint_as_float(l[0]) + __uint_as_float(l[1]);
                }
                acc[r][0][i] = f;
            }
    }
    // the waves' column ranges meet in LDS (each wave's sums in its own part, read by it alone until here),
    // summed in wave order; wave w stores tiles w, w + KW, ... (lane (c, g): row 16 r + c, tokens 16 t + 4 g .. + 3)
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int t = 0; t < TT; t++)
            *reinterpret_cast<f32x4*>(smem + wave * kLds + (r * TT + t) * 1024 + lane * 16) = acc[r][t];
    __syncthreads();
    for (int i = wave; i < R * TT; i += KW) {
        f32x4 v = *reinterpret_cast<const f32x4*>(smem + i * 1024 + lane * 16);
#pragma unroll
        for (int w = 1; w < KW; w++) v += *reinterpret_cast<const f32x4*>(smem + w * kLds + i * 1024 + lane * 16);
        const int row = r0 + 16 * (i / TT) + c, tok = t0 + 16 * (i % TT) + 4 * g;
        if (row >= a.rows) continue;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float y = v[e];
            if (a.post == 1) {
                const float u = y * a.post_scale;
                y = u / (1.0f + __expf(-u));
            }
            if (tok + e < a.n) a.y[(size_t)(tok + e) * a.y_stride + row] = y;
        }
    }
}

template <int TT, int R, int NS, int B, int KW>
constexpr size_t tok_lds() {
    return KW * (sizeof(TokLds<TT, R, NS, B>) > R * TT * 1024 ? sizeof(TokLds<TT, R, NS, B>) : R * TT * 1024);
}

// Grid (row groups of every matrix in turn, token groups)
template <int TT, int R, int NS, int B, int KW>
__global__ __launch_bounds__(64 * KW) void k_mat_tok(MatMultiArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    int i = 0;
    while (i + 1 < a.count && (int)blockIdx.x >= a.wg_end[i]) i++;
    mat_tok_body<TT, R, NS, B, KW>(a.m[i], (int)blockIdx.x - (i ? a.wg_end[i - 1] : 0), blockIdx.y, smem);
}

template <int BN>
__global__ __launch_bounds__(256, 2) void k_gemm(MatArgs a) {
    constexpr int NT = BN / 32;                      // 16-token tiles a wave (BN = 32, 64 or 128)
    constexpr int W_B = kGemmBM * 64;                // one bf16 weight plane of a stage
    constexpr int X_B = BN * 64;                     // one bf16 token plane
    constexpr int STAGE = 2 * W_B + 2 * X_B;
    __shared__ __attribute__((aligned(16))) unsigned char smem[2 * STAGE];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c = lane & 15, g = lane >> 4;
    const int wr = wave & 1, wt = wave >> 1;

    const int RT = (a.rows + kGemmBM - 1) / kGemmBM, TT = (a.n + BN - 1) / BN, T = RT * TT;
    const int b = blockIdx.x;
    const int idx = (T & 7) ? b : (b & 7) * (T >> 3) + (b >> 3);  // XCD b % 8 takes tiles [x T/8, (x+1) T/8)
    const int r0 = (idx / TT) * kGemmBM, t0 = (idx % TT) * BN;
    const int nkb = a.cols >> 5;

    // loader roles: weight row lr (two threads a row, 16 columns each); token row lt
    const int lr = tid >> 1, lh = tid & 1;
    const size_t wrow = (size_t)min(r0 + lr, a.rows - 1);
    constexpr int XT = BN >= 64 ? 256 / BN : 4;       // threads a token row (2 or 4)
    constexpr int XC = 32 / XT;                       // columns a thread (16 or 8)
    const int lt = tid / XT, lq = tid % XT;
    const bool xl = BN * XT == 256 || tid < BN * XT;  // BN = 32: threads 0..127 load the token rows
    const float* xrow = a.x + (size_t)min(t0 + min(lt, BN - 1), a.n - 1) * a.x_stride + lq * XC;

    // one step's global data in registers
    struct Pre {
        float f[16];   // weights
        float x[XC];
    };
    auto load = [&](Pre& P, int kb) {
        const int k0 = kb * 32;
        const float* wp = static_cast<const float*>(a.w) + wrow * a.cols + k0 + 16 * lh;
#pragma unroll
        for (int i = 0; i < 16; i += 4) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(wp + i);
            P.f[i] = v[0], P.f[i + 1] = v[1], P.f[i + 2] = v[2], P.f[i + 3] = v[3];
        }
        if (xl) {
#pragma unroll
            for (int i = 0; i < XC; i += 4) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(xrow + k0 + i);
                P.x[i] = v[0], P.x[i + 1] = v[1], P.x[i + 2] = v[2], P.x[i + 3] = v[3];
            }
        }
    };
    auto store = [&](const Pre& P, int st) {
        unsigned char* S = smem + st * STAGE;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            float v8[8];
#pragma unroll
            for (int j = 0; j < 8; j++) v8[j] = P.f[8 * h + j];
            bf16x8 hi, lo;
            split_bf16(v8, hi, lo);
            *reinterpret_cast<bf16x8*>(S + gemm_off(lr, 2 * lh + h)) = hi;
            *reinterpret_cast<bf16x8*>(S + W_B + 2 * X_B + gemm_off(lr, 2 * lh + h)) = lo;
        }
#pragma unroll
        for (int h = 0; h < XC / 8; h++) {
            if (!xl) break;
            float v8[8];
#pragma unroll
            for (int j = 0; j < 8; j++) v8[j] = P.x[8 * h + j];
            bf16x8 hi, lo;
            split_bf16(v8, hi, lo);
            const int gc = lq * (XC / 8) + h;
            *reinterpret_cast<bf16x8*>(S + W_B + gemm_off(lt, gc)) = hi;
            *reinterpret_cast<bf16x8*>(S + W_B + X_B + gemm_off(lt, gc)) = lo;
        }
    };

    f32x4 acc[4][NT];
#pragma unroll
    for (int m = 0; m < 4; m++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    auto compute = [&](int st) {
        const unsigned char* S = smem + st * STAGE;
        bf16x8 A[4], Bh[NT], Bl[NT];
#pragma unroll
        for (int m = 0; m < 4; m++) A[m] = *reinterpret_cast<const bf16x8*>(S + gemm_off(wr * 64 + m * 16 + c, g));
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int r = wt * (BN / 2) + t * 16 + c;
            Bh[t] = *reinterpret_cast<const bf16x8*>(S + W_B + gemm_off(r, g));
            Bl[t] = *reinterpret_cast<const bf16x8*>(S + W_B + X_B + gemm_off(r, g));
        }
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const bf16x8 Al = *reinterpret_cast<const bf16x8*>(S + W_B + 2 * X_B + gemm_off(wr * 64 + m * 16 + c, g));
#pragma unroll
            for (int t = 0; t < NT; t++) {
                acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[m], Bh[t], acc[m][t], 0, 0, 0);
                acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[m], Bl[t], acc[m][t], 0, 0, 0);
                acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Al, Bh[t], acc[m][t], 0, 0, 0);
                acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Al, Bl[t], acc[m][t], 0, 0, 0);
            }
        }
    };

    // stage kb % 2 holds step kb; step kb + 1's global loads are in flight while its MFMAs run, then
    // converted into the other stage (whose last readers passed the previous barrier)
    Pre P;
    load(P, 0);
    store(P, 0);
    __syncthreads();
    for (int kb = 0; kb < nkb; kb++) {
        if (kb + 1 < nkb) load(P, kb + 1);
        compute(kb & 1);
        if (kb + 1 < nkb) store(P, (kb + 1) & 1);
        __syncthreads();
    }

    // lane (c, g) holds rows 4 g .. 4 g + 3 of each tile for token c
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int tok = t0 + wt * (BN / 2) + t * 16 + c;
        if (tok >= a.n) continue;
        float* yr = a.y + (size_t)tok * a.y_stride;
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const int row = r0 + wr * 64 + m * 16 + 4 * g;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float v = acc[m][t][i];
                if (a.post == 1) {
                    const float u = v * a.post_scale;
                    v = u / (1.0f + __expf(-u));
                }
                if (row + i < a.rows) yr[row + i] = v;
            }
        }
    }
}

// ---- Q8, many tokens: tiled MFMA GEMM ---------------------------------------------------------------
// Replaces the q4_gemm_q8 pipeline (shaders/q4_gemm.comp) that Qwen4Vulkan::mat selects from nine tokens on
// (src/qwen4_vk.cpp:852-853).
// A workgroup of eight waves owns a tile of BM = 32 RT GR rows x BN = 32 TT GT tokens, each wave 32 RT x 32 TT of
// it, and walks the columns 64 (two Q8 blocks) at a time through two LDS stages: per 32-column block and 32 x 32
// piece four v_mfma_f32_32x32x16_bf16 (two column halves of the hi, then of the lo part of x; the weights exact
// in bf16, the B operand) into a fresh accumulator that is scaled by the lane's row's block scale into the
// running sum.
//
// What bounds it is a SIMD's issue: per MFMA eight other vector instructions (half of them the scaling, the rest
// the conversion of int8 and fp32 to bf16), and the two share it: 32x32x16 with eight of them 18.7 ns (14.2 with
// none), 16x16x32, half the work, with four 14.4 ns (8.3 with none). Then the step's barrier and operand reads,
// which both waves of a SIMD wait for together. 8,192 x 2,048 at 2,048 tokens, one box: 200 us with 128 x 128
// tiles of four waves a workgroup and token rows loaded two lanes a row; 148 with rows loaded by consecutive
// lanes and 256 x 128 tiles, alike with 16x16x32 MFMAs in the compiler's order or pinned; 147 with 32x32x16, of
// which the conversions take 30 and the scaling, by leaving three quarters of it out, 18.
template <int RT, int TT, int GR, int GT>
__global__ __launch_bounds__(512, RT * TT == 1 ? 4 : 2) void k_gemm_q8(MatArgs a) {
    static_assert(GR * GT == 8, "eight waves");
    constexpr int BM = 32 * RT * GR, BN = 32 * TT * GT;
    constexpr int WL = BM / 128, XL = BN / 32;  // 16-byte loads a thread and step: weights, token rows
    constexpr int W_B = BM * 128, X_B = BN * 128, STAGE = W_B + 2 * X_B + BM * 8;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int c = lane & 31, h = lane >> 5;
    const int wr = (wave % GR) * 32 * RT, wt = (wave / GR) * 32 * TT;

    const int RTs = (a.rows + BM - 1) / BM, TTs = (a.n + BN - 1) / BN, T = RTs * TTs;
    const int b = blockIdx.x;
    const int idx = (T & 7) ? b : (b & 7) * (T >> 3) + (b >> 3);  // XCD b % 8 takes tiles [x T/8, (x+1) T/8)
    const int r0 = (idx / TTs) * BM, t0 = (idx % TTs) * BN;
    const int nkb = a.cols >> 5, nst = (nkb + 1) >> 1;

    // loads by consecutive lanes: four lanes a weight row's 64 columns, sixteen a token's. Rows and tokens past the
    // ends, and a last half step's second block, lie outside the resources and read zero: the whole offset is in the
    // per-lane operand, since the range check leaves the scalar offset out. The additions cost nothing at 8,192 x
    // 2,048 (2,048 tokens 152-154 us with the rows and steps in the scalar offset, 152 without) and 0.3-2 us of 92 and 55
    // at 2,048 x 4,096 (2,048 and 1,024 tokens).
    const int wq = tid & 3, xq = tid & 15;
    const int nr = min(BM, a.rows - r0), nt = min(BN, a.n - t0);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int8_t*>(static_cast<const int8_t*>(a.w)) + (size_t)r0 * a.cols, (short)0, nr * a.cols, 0x00020000);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(a.s) + (size_t)r0 * nkb, (short)0, nr * nkb * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(a.x) + (size_t)t0 * a.x_stride, (short)0, ((nt - 1) * a.x_stride + a.cols) * 4, 0x00020000);
    u32x4 wv[WL];
    f32x4 xv[XL];
    float sv;
    auto load_w = [&](int k) {
#pragma unroll
        for (int i = 0; i < WL; i++)
            wv[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                rw, (int)gemm_w_off(128 * i + (tid >> 2), wq, k, a.cols, nkb), 0, 0));
        sv = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, (int)gemm_s_off((tid >> 1) % BM, tid & 1, k, nkb), 0, 0));
    };
    auto load_x = [&](int k, int i) {
        xv[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
            rx, (int)gemm_x_off(32 * i + (tid >> 4), xq, k, a.x_stride, nkb), 0, 0));
    };
    // LDS rows of 64 columns are eight 16-byte chunks, chunk q of row r at q ^ (r / 2) % 8, which spreads operand reads
    // (16 rows' chunk q) and the loaders' writes over the banks: conflicts are 0.17 of the LDS's active cycles (256 x
    // 128 tiles), and waves wait for it 5% of theirs
    auto at = [](int r, int q) { return r * 128 + ((q ^ ((r >> 1) & 7)) << 4); };
    // the conversion of the loaded pieces in units of a few instructions: four to each half of a weight piece (its
    // pairs of weights), two to a token piece
    constexpr int UW = 8 * WL, U = UW + 2 * XL;
    uint32_t cw[4], ch[2], cl[2];
    auto unit = [&](int u, unsigned char* S) {
        if (u < UW) {
            const int i = u / 8, hf = u / 4 % 2, e = u % 4;
            const int v = (int)wv[i][2 * hf + e / 2], sh = 16 * (e & 1);
            cw[e] = pk_bf16((float)((v << (24 - sh)) >> 24), (float)((v << (16 - sh)) >> 24));
            if (e == 3) *reinterpret_cast<u32x4*>(S + at(128 * i + (tid >> 2), 2 * wq + hf)) = u32x4{cw[0], cw[1], cw[2], cw[3]};
        } else {
            const int i = (u - UW) / 2, e = (u - UW) % 2;
            const float v0 = xv[i][2 * e], v1 = xv[i][2 * e + 1];
            ch[e] = pk_bf16(v0, v1);
            cl[e] = pk_bf16(rest_bf16<0>(ch[e], v0), rest_bf16<1>(ch[e], v1));
            if (e == 1) {
                unsigned char* d = S + W_B + at(32 * i + (tid >> 4), xq >> 1) + 8 * (xq & 1);
                *reinterpret_cast<u32x2*>(d) = u32x2{ch[0], ch[1]};
                *reinterpret_cast<u32x2*>(d + X_B) = u32x2{cl[0], cl[1]};
            }
        }
    };
    // (the scale of a block past the row reads as 0: a last half step's second block adds nothing)
    auto put_s = [&](unsigned char* S) {
        if (tid < 2 * BM) reinterpret_cast<float*>(S + W_B + 2 * X_B)[(tid & 1) * BM + (tid >> 1)] = sv;
    };

    f32x16 acc[RT][TT];
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = 0; t < TT; t++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[r][t][e] = 0.f;

    load_w(0);
#pragma unroll
    for (int i = 0; i < XL; i++) load_x(0, i);
#pragma unroll
    for (int u = 0; u < U; u++) unit(u, smem);
    put_s(smem);
    load_w(min(1, nst - 1));
#pragma unroll
    for (int i = 0; i < XL; i++) load_x(min(1, nst - 1), i);
    __syncthreads();
    // Stage k % 2 holds step k; while its MFMAs run, step k + 1 (loaded a step ago) is converted into the other
    // stage, whose last readers passed the previous barrier, and step k + 2's loads follow each piece. A step is
    // 2 TT RT passes (block j, token tile t, row tile r) of four slots: one MFMA, the scaling of a quarter of the
    // pass before, a conversion unit or so, pinned in this order so that a wave's MFMAs and its other
    // instructions take turns. The step past the last is converted too, unread.
    constexpr int P = 2 * TT * RT, SL = 4 * P;
    bf16x8 W[2][RT][2], xf[2][2][2];  // [block][row tile][column half]; [(j, t) parity][part][column half]
    float sc[2][RT];
    f32x16 d[2];
#pragma unroll
    for (int e = 0; e < 16; e++) d[1][e] = 0.f;
#pragma unroll
    for (int r = 0; r < RT; r++) sc[1][r] = 0.f;
#pragma unroll 1
    for (int k = 0; k < nst; k++) {
        const unsigned char* S = smem + (k & 1) * STAGE;
        unsigned char* N = smem + ((k + 1) & 1) * STAGE;
        const float* sS = reinterpret_cast<const float*>(S + W_B + 2 * X_B);
        const int k2 = min(k + 2, nst - 1);
        auto read_w = [&](int j, int r, int q) {
            W[j][r][q] = *reinterpret_cast<const bf16x8*>(S + at(wr + 32 * r + c, 4 * j + 2 * q + h));
        };
        auto read_x = [&](int jt, int part, int q) {
            xf[jt & 1][part][q] = *reinterpret_cast<const bf16x8*>(
                S + W_B + part * X_B + at(wt + 32 * (jt % TT) + c, 4 * (jt / TT) + 2 * q + h));
        };
#pragma unroll
        for (int q = 0; q < 2; q++) read_w(0, 0, q), read_x(0, 0, q);
#pragma unroll
        for (int q = 0; q < 2; q++) read_x(0, 1, q);
#pragma unroll
        for (int r = 1; r < RT; r++) read_w(0, r, 0), read_w(0, r, 1);
        static_for<0, SL>([&](auto s_) {
            constexpr int s = s_, p = s / 4, q4 = s % 4;
            constexpr int r = p % RT, jt = p / RT, t = jt % TT, j = jt / TT;
            constexpr int pp = (p + P - 1) % P, pr = pp % RT, pt = pp / RT % TT, pj = pp / RT / TT;  // the pass before
            constexpr int part = q4 / 2, q = q4 % 2;
            const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            d[p & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xf[jt & 1][part][q], W[j][r][q], q4 ? d[p & 1] : zero, 0, 0, 0);
            // (none in the first slot: the pass before's last MFMA has not ended yet)
            constexpr int f0 = q4 < 2 ? 0 : 5 * q4 - 4, f1 = q4 == 0 ? 0 : 5 * q4 + 1;
#pragma unroll
            for (int e = f0; e < f1; e++) {
                float v = __builtin_fmaf(sc[pj][pr], d[(p + 1) & 1][e], acc[pr][pt][e]);
                asm volatile("" : "+v"(v));  // here, not sunk to the step's end
                acc[pr][pt][e] = v;
            }
            // units: the pass's first two thirds in its first slot, the rest in its last
            constexpr int u0 = p * U / P, u2 = (p + 1) * U / P, u1 = u0 + (2 * (u2 - u0) + 2) / 3;
            static_for<q4 == 0 ? u0 : u1, q4 == 0 ? u1 : q4 == 3 ? u2 : u1>([&](auto u_) {
                constexpr int u = u_;
                unit(u, N);
                if constexpr (u == UW - 1) {
                    put_s(N);
                    load_w(k2);
                }
                if constexpr (u >= UW && (u - UW) % 2 == 1) load_x(k2, (u - UW) / 2);
            });
            // the next token tile's operands and the second block's weights ahead of their passes; the scales of
            // this step's blocks once the last pass of the step before has used its own
            if constexpr (r == RT - 1 && jt + 1 < 2 * TT) read_x(jt + 1, q4 / 2, q4 % 2);
            if constexpr (j == 0 && t == TT - 1 && q4 < 2) read_w(1, r, q4);
            if constexpr (p == 0 && q4 == 3) {
#pragma unroll
                for (int i = 0; i < RT; i++) sc[0][i] = sS[wr + 32 * i + c], sc[1][i] = sS[BM + wr + 32 * i + c];
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        __syncthreads();
    }
#pragma unroll
    for (int e = 0; e < 16; e++)
        acc[RT - 1][TT - 1][e] = __builtin_fmaf(sc[1][RT - 1], d[1][e], acc[RT - 1][TT - 1][e]);

    // lane (c, h): row 32 r + c of the wave's, tokens 32 t + 8 (e / 4) + 4 h + e % 4
#pragma unroll
    for (int t = 0; t < TT; t++)
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int tok = t0 + wt + 32 * t + 8 * (e / 4) + 4 * h + e % 4;
            if (tok >= a.n) continue;
            float* yr = a.y + (size_t)tok * a.y_stride;
#pragma unroll
            for (int r = 0; r < RT; r++) {
                const int row = r0 + wr + 32 * r + c;
                float v = acc[r][t][e];
                if (a.post == 1) {
                    const float u = v * a.post_scale;
                    v = u / (1.0f + __expf(-u));
                }
                if (row < a.rows) yr[row] = v;
            }
        }
}

template <int RT, int TT, int GR, int GT>
constexpr size_t gemm_lds() {
    return 2 * (32 * RT * GR * 136 + 2 * 32 * TT * GT * 128);
}

}  // namespace

namespace {

constexpr int kTokGroups = 65535;  // token groups a launch

template <int TT, int R, int NS, int B, int KW>
hipError_t launch_tok(MatMultiArgs a, hipStream_t s) {
    constexpr size_t lds = tok_lds<TT, R, NS, B, KW>();
    static std::atomic<uint64_t> raised{0};
    if (const hipError_t e = raise_lds((const void*)k_mat_tok<TT, R, NS, B, KW>, lds, raised); e != hipSuccess) return e;
    int wg = 0;
    for (int i = 0; i < a.count; i++) a.wg_end[i] = wg += (a.m[i].rows + 16 * R - 1) / (16 * R);
    // as many launches as the grid's y limit asks for
    const int n = a.m[0].n, most = kTokGroups * 16 * TT;
    for (int t0 = 0;;) {
        const int nt = std::min(most, n - t0);
        for (int i = 0; i < a.count; i++) a.m[i].n = nt;
        hipLaunchKernelGGL((k_mat_tok<TT, R, NS, B, KW>), dim3(wg, (nt + 16 * TT - 1) / (16 * TT)), dim3(64 * KW), lds, s, a);
        if (const hipError_t e = hipGetLastError(); e != hipSuccess || n - t0 == nt) return e;
        t0 += nt;
        for (int i = 0; i < a.count; i++) a.m[i].x += (size_t)nt * a.m[i].x_stride, a.m[i].y += (size_t)nt * a.m[i].y_stride;
    }
}

// The token-tile kernel's shapes with two parts a token value. Eight waves (a workgroup a CU) up to 64 tokens, or
// from 4,096 columns; four (two workgroups a CU) otherwise: 9,216 x 2,048 at 64 / 80 / 256 tokens 16.6 / 23.7 /
// 56 us with eight, 18.9 / 20.5 / 46 with four; 2,048 x 4,096 at 80 / 256 14.2 / 20.6 and 16.0 / 23.9. The wave
// count decides the order of a sum, so it depends on nothing that differs between qwattn_mat and
// qwattn_mat_multi; the tile counts do not.
struct TokShape {
    int tt, r;
    hipError_t (*launch)(MatMultiArgs, hipStream_t);
};
constexpr TokShape kTok8[] = {{1, 1, launch_tok<1, 1, 2, 1, 8>}, {1, 2, launch_tok<1, 2, 2, 1, 8>},
                              {1, 3, launch_tok<1, 3, 2, 1, 8>}, {1, 4, launch_tok<1, 4, 2, 1, 8>},
                              {2, 2, launch_tok<2, 2, 2, 1, 8>}, {2, 3, launch_tok<2, 3, 2, 1, 8>},
                              {2, 4, launch_tok<2, 4, 2, 1, 8>}, {3, 2, launch_tok<3, 2, 2, 1, 8>},
                              {3, 3, launch_tok<3, 3, 2, 1, 8>}, {3, 4, launch_tok<3, 4, 2, 1, 8>},
                              {4, 3, launch_tok<4, 3, 2, 1, 8>}};
constexpr TokShape kTok4[] = {{1, 2, launch_tok<1, 2, 2, 1, 4>}, {1, 4, launch_tok<1, 4, 2, 1, 4>},
                              {2, 4, launch_tok<2, 4, 2, 1, 4>}};
constexpr int kCus = 256;

// Row groups of 16 R rows, every matrix by itself.
int row_groups(const MatMultiArgs& a, int r) {
    int g = 0;
    for (int i = 0; i < a.count; i++) g += (a.m[i].rows + 16 * r - 1) / (16 * r);
    return g;
}

// Whether the token-tile kernel's 32-bit offsets reach every operand (up to 64 rows and tokens a workgroup).
bool tok_fits(const MatMultiArgs& a) {
    const MatArgs& m = a.m[0];
    return m.cols <= 1 << 24 && (63ll * m.x_stride + m.cols) * 4 < kFar;
}

hipError_t launch_tok_any(const MatMultiArgs& a, hipStream_t s) {
    const MatArgs& m = a.m[0];
    if (m.n < 16) {
        // as many row tiles a workgroup as leave a workgroup a CU, three at most (9,216 x 2,048 at 12 tokens: one
        // tile 13.1 us, two 12.2, three 9.9, four 11.2)
        const int r = row_groups(a, 1) <= kCus ? 1 : row_groups(a, 2) <= kCus ? 2 : 3;
        if (m.n <= 4)
            return r == 1 ? launch_tok<1, 1, 3, 4, 8>(a, s) : r == 2 ? launch_tok<1, 2, 3, 4, 8>(a, s) : launch_tok<1, 3, 3, 4, 8>(a, s);
        if (m.n <= 8)
            return r == 1 ? launch_tok<1, 1, 3, 2, 8>(a, s) : r == 2 ? launch_tok<1, 2, 3, 2, 8>(a, s) : launch_tok<1, 3, 3, 2, 8>(a, s);
        return r == 1 ? launch_tok<1, 1, 3, 1, 8>(a, s) : r == 2 ? launch_tok<1, 2, 3, 1, 8>(a, s) : launch_tok<1, 3, 3, 1, 8>(a, s);
    }
    const int tiles = (m.n + 15) / 16;
    const auto wgs = [&](const TokShape& k) { return row_groups(a, k.r) * ((tiles + k.tt - 1) / k.tt); };
    if (m.n <= 64 || m.cols >= 4096) {
        // instructions a block: splitting and laying out a token tile, converting a row tile, the product of both
        const TokShape* best = nullptr;
        long long least = 0;
        for (const TokShape& k : kTok8) {
            const long long t = (long long)((wgs(k) + kCus - 1) / kCus) * (30 * k.tt + 14 * k.r + 8 * k.tt * k.r);
            if (!best || t < least) best = &k, least = t;
        }
        return best->launch(a, s);
    }
    // the largest shape that still gives every CU a workgroup
    const TokShape* k = &kTok4[2];
    while (k > kTok4 && wgs(*k) < kCus) k--;
    return k->launch(a, s);
}

template <int RT, int TT, int GR, int GT>
hipError_t launch_gemm_q8(const MatArgs& a, hipStream_t s) {
    constexpr size_t lds = gemm_lds<RT, TT, GR, GT>();
    static std::atomic<uint64_t> raised{0};
    if (const hipError_t e = raise_lds((const void*)k_gemm_q8<RT, TT, GR, GT>, lds, raised); e != hipSuccess) return e;
    const int bm = 32 * RT * GR, bn = 32 * TT * GT;
    hipLaunchKernelGGL((k_gemm_q8<RT, TT, GR, GT>), dim3(((a.rows + bm - 1) / bm) * ((a.n + bn - 1) / bn)), dim3(512), lds, s, a);
    return hipGetLastError();
}

// The Q8 GEMM's tiles with what a 64-column step of one takes a CU, in hundredths of a microsecond (one tile a CU;
// 2,048 tokens through 8,192 x 2,048 and 2,048 x 4,096: 147 / 184 / 213 and 107 / 86 / 107 us).
struct GemmTile {
    int bm, bn, step;
    hipError_t (*launch)(const MatArgs&, hipStream_t);
};
constexpr GemmTile kGemmTiles[] = {{256, 128, 235, launch_gemm_q8<2, 2, 4, 2>},
                                   {128, 128, 135, launch_gemm_q8<2, 1, 2, 4>},
                                   {128, 64, 82, launch_gemm_q8<1, 1, 4, 2>}};
int gemm_cost(const GemmTile& t, int rows, int n) {
    const long long tiles = (long long)((rows + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn);
    return (int)std::min<long long>((tiles + kCus - 1) / kCus * t.step, 1 << 30);
}
const GemmTile& gemm_tile(int rows, int n) {
    const GemmTile* best = kGemmTiles;
    for (const GemmTile& t : kGemmTiles)
        if (gemm_cost(t, rows, n) < gemm_cost(*best, rows, n)) best = &t;
    return *best;
}
// Whether the Q8 GEMM's 32-bit offsets reach the operands.
bool gemm_fits(const MatArgs& a) { return gemm_offsets_fit(a.cols, a.x_stride); }

// Whether a Q8 matrix takes the token-tile kernel (from two tokens on): up to 64 tokens, else where its 64-row x
// 32-token workgroups, two a CU and 0.55 us a pair and 64 columns, take less than the GEMM's tiles (8,192 x 2,048
// at 128 / 256 / 512 tokens 21 / 37 / 68 us against 29 / 31 / 46; 2,048 x 4,096 at 256 / 512 / 777 22 / 39 / 66
// against 50 / 51 / 52; 512 x 2,048 at 2,048 27 against 29). By the matrix alone, so that qwattn_mat and
// qwattn_mat_multi agree. For the same reason a small matrix called by itself with 2 to 15 tokens stays here although a
// matrix-vector kernel of fp32 multiply-adds is faster then (256 x 2,048 at 4 / 8 / 15 tokens 5.2 / 6.2 / 7.2 us, 4.6 /
// 4.7 / 4.7): beside a larger one in qwattn_mat_multi it costs this kernel next to nothing, but on matrix-vector
// workgroups in the same launch 8,192 + 512 + 512 rows of 2,048 columns went from 11.4 / 11.9 us at 4 / 8 tokens to
// 12.6 / 15.1.
bool tok_wins(const MatArgs& a) {
    if (a.n <= 64) return true;
    const long long wgs = (long long)((a.rows + 63) / 64) * ((a.n + 31) / 32);
    return std::max<long long>(55, 55 * wgs / (2 * kCus)) <= gemm_cost(gemm_tile(a.rows, a.n), a.rows, a.n);
}

}  // namespace

hipError_t launch_mat(const MatArgs& a, bool q8, hipStream_t s) {
    if (q8 && a.n > 1) {
        MatMultiArgs m{};
        m.m[0] = a, m.count = 1;
        const bool gemm = gemm_fits(a);
        if (tok_fits(m) && (!gemm || tok_wins(a))) return launch_tok_any(m, s);
        if (gemm) return gemm_tile(a.rows, a.n).launch(a, s);
    }
    if (!q8 && a.n >= kGemmMinN && a.cols % 32 == 0) {
        // the widest token tile that still gives two workgroups a CU (fewer weight re-reads), else the
        // narrowest (the most workgroups)
        const int rt = (a.rows + kGemmBM - 1) / kGemmBM;
        const auto tiles = [&](int bn) { return rt * ((a.n + bn - 1) / bn); };
        const int bn = tiles(128) >= 512 ? 128 : tiles(64) >= 512 ? 64 : 32;
        const dim3 grid(tiles(bn)), block(256);
        if (bn == 128) hipLaunchKernelGGL((k_gemm<128>), grid, block, 0, s, a);
        else if (bn == 64) hipLaunchKernelGGL((k_gemm<64>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((k_gemm<32>), grid, block, 0, s, a);
        return hipGetLastError();
    }
    // matrix-vector: one token a workgroup for a decode step and for Q8 (whose other token counts come here only
    // with row strides past the token-tile kernel's offsets), else four; four rows a wave when that still gives
    // 256 workgroups a token group, else one (small matrices: more rows in flight at once)
    const int ntp = q8 || a.n == 1 ? 1 : kMatNTP;
    const bool rw4 = a.rows >= 4096;
    if ((a.n + ntp - 1) / ntp > 65535) return hipErrorInvalidConfiguration;  // grid y limit (f32, cols % 32 != 0)
    const dim3 grid((a.rows + (rw4 ? 15 : 3)) / (rw4 ? 16 : 4), (a.n + ntp - 1) / ntp), block(256);
    if (q8) {
        if (rw4) hipLaunchKernelGGL((k_mat_q8<4>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((k_mat_q8<1>), grid, block, 0, s, a);
    } else if (ntp == 1) {
        if (rw4) hipLaunchKernelGGL((k_mat_f32<1, 4>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((k_mat_f32<1, 1>), grid, block, 0, s, a);
    } else {
        if (rw4) hipLaunchKernelGGL((k_mat_f32<kMatNTP, 4>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((k_mat_f32<kMatNTP, 1>), grid, block, 0, s, a);
    }
    return hipGetLastError();
}

hipError_t launch_mat_multi(const MatMultiArgs& a0, bool q8, hipStream_t s) {
    const MatArgs& f = a0.m[0];
    if ((q8 && f.n > 1) || (f.n >= kGemmMinN && f.cols % 32 == 0)) {
        // the matrices that the token-tile kernel takes in one launch, the GEMM's by themselves (each fills the
        // chip)
        MatMultiArgs t{};
        for (int i = 0; i < a0.count; i++) {
            if (q8 && tok_fits(a0) && (tok_wins(a0.m[i]) || !gemm_fits(f))) {
                t.m[t.count++] = a0.m[i];
            } else if (const hipError_t e = launch_mat(a0.m[i], q8, s); e != hipSuccess) {
                return e;
            }
        }
        return t.count ? launch_tok_any(t, s) : hipSuccess;
    }
    MatMultiArgs a = a0;
    int rows = 0;
    for (int i = 0; i < a.count; i++) rows += a.m[i].rows;
    const int ntp = f.n == 1 ? 1 : kMatNTP;
    const bool rw4 = rows >= 4096;
    if ((f.n + ntp - 1) / ntp > 65535) return hipErrorInvalidConfiguration;  // grid y limit (f32, cols % 32 != 0)
    int wg = 0;
    for (int i = 0; i < a.count; i++) {
        wg += (a.m[i].rows + (rw4 ? 15 : 3)) / (rw4 ? 16 : 4);
        a.wg_end[i] = wg;
    }
    const dim3 grid(wg, (f.n + ntp - 1) / ntp), block(256);
#define QW_MULTI(Q, N, R) hipLaunchKernelGGL((k_mat_multi<Q, N, R>), grid, block, 0, s, a)
    if (q8) {
        if (rw4) QW_MULTI(true, 1, 4);
        else QW_MULTI(true, 1, 1);
    } else {
        if (ntp == 1) { if (rw4) QW_MULTI(false, 1, 4); else QW_MULTI(false, 1, 1); }
        else { if (rw4) QW_MULTI(false, kMatNTP, 4); else QW_MULTI(false, kMatNTP, 1); }
    }
#undef QW_MULTI
    return hipGetLastError();
}

}  // namespace qw
