// Batched prefill of a prompt: the reference runs a prompt one token at a
// time through the decode layers (HybridModel::prefill,
// nexus/src/model/hybrid_model.cpp:604-644); here a chunk of P prompt tokens
// goes through each layer at once, so every projection is a GEMM
// [P x K] x [K x N] on the matrix cores instead of P weight-streaming GEMVs.
//
// k_pf_gemm: Y = X W^T with X fp16 [M][ldx] (tokens) and W int4-g32 (codes
// [N][G*16], fp16 scales [N][G]).  A block computes 32 NI WM tokens x 256
// weight rows; each wavefront takes 32 NI tokens x 64 weight rows in tiles of
// v_mfma_f32_32x32x16_f16 (A = X: row = token; B = W: column = weight row).
// Exact scaling: the codes enter as (q - 8) 2^-9, a group's two products
// give its sum over 32 k, and one fp32 fma per output multiplies it by the
// group's scale into the accumulator (the sums are of exact products; 2^9 is
// applied at the end).  What bounds it: the matrix cores and the vector ALU
// of a SIMD hardly overlap (a 32 x 32 x 16 product and 8 fmas take 41 cycles
// together at two wavefronts, 32 and 17 alone; two 16 x 16 x 32 products and
// the same fmas take 50), so a SIMD's time is the products (64 cycles per
// 32 x 32 tile and group), the scale fmas (16 at 2.2 cycles) and the code
// conversion (8 permutes and 8 packed fmas at 4.4, 6 logic operations, once
// per 128 tokens), about 1.55 PFLOP/s at 2.4 GHz; the full chip holds less
// than that clock.  (The scheme before split each scale into two parts
// exact in fp16 and paid two products per group: 575 TFLOP/s at M 2048,
// N 28672, K 4096, and twice this one's rounding error; now 915.)
// X, codes and scales go to LDS without registers, X three stages of 64 k
// deep, codes and scales two of 128 k; the one barrier of a stage stands in
// its middle, a stage's operands are read from LDS during the stage before,
// and the products of one 32 x 32 tile run ahead of the previous tile's
// fmas, so a wavefront waits for neither memory nor LDS nor a product.
// (Barriers at the stage's ends and operands read after them: 580 us instead
// of 524 at that size; requests made through the compiler's builtin, which
// then waits for them before every LDS read: 593.)
// Epilogues: fp32 store, fp32 accumulate (residual), SwiGLU of interleaved
// gate/up rows to fp16; products with too few tiles for the chip split K,
// their part sums meet in k_pf_ksum.
#include <algorithm>
#include <type_traits>

#include "nx_common.h"
#include "nx_kernels.h"

namespace nx {
namespace {

typedef _Float16 ph8_t __attribute__((ext_vector_type(8)));
typedef float pf16_t __attribute__((ext_vector_type(16)));

constexpr int kPfThreads = 256;
constexpr int kPfXcds = 8;  // blocks are dealt to the XCDs round-robin by block index
constexpr int kPfBN = 256, kPfBK = 64;  // weight rows per block (64 per wavefront), k per stage (two groups)

// Pair h (k = 2h, 2h + 1) of a code dword (8 nibbles, low nibble = even k) as
// fp16 (q - 8) 2^-9: each nibble, alone in a half, is the fp16 subnormal
// q 2^-24, and one packed fma gives q 2^-9 - 8 2^-9 exactly.
template <int h>
__device__ inline uint32_t pf_code_pair(uint32_t lo, uint32_t hi) {
    const half2_t q = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(hi, lo, 0x0C040C00u + 0x00010001u * h));
    const half2_t up = {(_Float16)32768.0f, (_Float16)32768.0f}, off = {(_Float16)-0.015625f, (_Float16)-0.015625f};
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(q, up, off));
}

__device__ inline float lane_xor1(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, false));
}

// silu(g) u in fp16: hardware exp and reciprocal (a few ulp in fp32, below
// the fp16 rounding of the stored activation)
__device__ inline uint16_t pf_swiglu(float g, float u) {
    return f2h_bits(g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) * u);
}

struct PfTiles {
    int ntm, ntn, ksplit;  // token tiles, weight-row tiles, K parts
    int sper;              // stages per K part
};

// WM x 4 wavefronts, each 32 NI tokens by 64 weight rows (NI 32-token tiles).
// FAST: K a multiple of 128 (no chunk past K, stages in pairs, a row's scales
// of 4 groups one aligned 8-byte load) and 32-bit offsets within a tile.
template <int EPI, int WM, int NI, bool FAST>
__global__ __launch_bounds__(kPfThreads * WM, 2) void k_pf_gemm(PfGemmArgs a, PfTiles tl) {
    constexpr int BM = 32 * NI * WM, NW = 4 * WM;
    constexpr int kXReq = BM / 8 / NW, kWReq = 16 / NW;  // 1 KiB requests per wavefront: of an X stage, of two stages' codes
    __shared__ __align__(16) uint4 Xs[3 * BM * 8];       // [buffer][row][8 chunks of 8 k], chunk ch in slot ch ^ (row & 7)
    __shared__ __align__(16) uint4 Ws[2 * 4 * kPfBN];    // [buffer][row][4 groups], group g in slot g ^ (row / 4 % 4)
    __shared__ __align__(16) uint2 Ss[2 * kPfBN];        // [buffer][row]: the 4 groups' fp16 scales
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave & 3, wm = wave >> 2;
    const int c = lane & 31, kh = lane >> 5;
    const int M = a.M, N = a.N, K = a.K, G = a.G;
    // XCD-aware tile order: XCD x (block index % 8 == x) takes an eighth of
    // the tiles in an order that walks K parts, then groups of 4 token
    // tiles, then weight-row tiles, then the group's token tiles, so the
    // blocks an XCD runs together share a few tiles of each operand in its L2
    const unsigned per = (unsigned)tl.ntm * tl.ntn, T = per * tl.ksplit;
    const unsigned xcd = blockIdx.x % kPfXcds, local = blockIdx.x / kPfXcds;
    const unsigned t0 = (unsigned)((unsigned long long)xcd * T / kPfXcds);
    if (local >= (unsigned)((unsigned long long)(xcd + 1) * T / kPfXcds) - t0) return;
    const unsigned idx = t0 + local, ks = idx / per, r0 = idx - ks * per;
    const unsigned mg = r0 / (4u * tl.ntn), gm = min(4u, tl.ntm - 4u * mg), rr = r0 - mg * 4u * tl.ntn;
    const int n0 = (int)(rr / gm) * kPfBN, m0 = (int)(4u * mg + rr % gm) * BM;
    const int nstage = (G + 1) / 2, sb = (int)ks * tl.sper, se = min(nstage, sb + tl.sper);
    if (sb >= se) return;

    // This lane's part of a stage: chunk (lane % 8) ^ (lane / 8) of one X row
    // per request (8 lanes read 128 contiguous bytes).  Codes and scales come
    // two stages (4 groups) at a time: 4 lanes read the 64 contiguous bytes of
    // a row's 4 groups (two groups at a time use 32 bytes of every 128-byte
    // line a request opens, and the L1 does not hold the lines for the next
    // stage).  Addresses past an edge are clamped into the tensor.
    const int xch = (lane & 7) ^ (lane >> 3), wg = (lane & 3) ^ (lane >> 4);
    using Off = std::conditional_t<FAST, uint32_t, size_t>;  // byte offsets from the tile's first row
    const char* xbase = reinterpret_cast<const char*>(a.x + (size_t)m0 * a.ldx);
    const uint8_t* wbase = a.W + (size_t)n0 * G * 16;
    Off xoff[kXReq], woff[kWReq];
#pragma unroll
    for (int j = 0; j < kXReq; ++j)
        xoff[j] = (Off)min(8 * (wave + NW * j) + (lane >> 3), M - 1 - m0) * (Off)(2 * a.ldx) + 16 * xch;
#pragma unroll
    for (int j = 0; j < kWReq; ++j)
        woff[j] = ((Off)min(16 * (wave + NW * j) + (lane >> 2), N - 1 - n0) * (Off)G + wg) * 16;
    auto load_x = [&](int s, int buf, int j) {
        const char* base = xbase + (size_t)s * (2 * kPfBK);
        // the last chunk again for chunks past K (zeroed by zero_x)
        const uint32_t back = FAST || (s + 1) * kPfBK <= K ? 0u : 2u * (uint32_t)max(s * kPfBK + 8 * xch - (K - 8), 0);
        dma16_lds(base, (Off)(xoff[j] - back), &Xs[buf * (BM * 8) + 64 * (wave + NW * j)]);
    };
    auto zero_x = [&](int s, int buf) {  // zeros over this wavefront's landed chunks past K
        if ((s + 1) * kPfBK > K && s * kPfBK + 8 * xch >= K)
#pragma unroll
            for (int j = 0; j < kXReq; ++j) Xs[buf * (BM * 8) + 64 * (wave + NW * j) + lane] = make_uint4(0, 0, 0, 0);
    };
    const uint16_t* sp = a.S + (size_t)min(n0 + (tid & (kPfBN - 1)), N - 1) * G;
    uint2 rs = make_uint2(0, 0);
    auto load_w = [&](int s, int buf, int j) {  // s: the first of the two stages
        const uint8_t* base = wbase + (size_t)(2 * s) * 16;
        const uint32_t back = FAST ? 0u : 16u * (uint32_t)max(2 * s + wg - (G - 1), 0);
        dma16_lds(base, (Off)(woff[j] - back), &Ws[buf * (4 * kPfBN) + 64 * (wave + NW * j)]);
    };
    auto load_s = [&](int s) {
        if (WM == 1 || wave < 4) {
            if (FAST) {
                rs = *reinterpret_cast<const uint2*>(sp + 2 * s);
            } else {
                rs.x = sp[2 * s] | (uint32_t)sp[min(2 * s + 1, G - 1)] << 16;
                rs.y = sp[min(2 * s + 2, G - 1)] | (uint32_t)sp[min(2 * s + 3, G - 1)] << 16;
            }
        }
    };
    auto store_s = [&](int buf) {
        if (WM == 1 || wave < 4) Ss[buf * kPfBN + tid] = rs;
    };

    pf16_t acc[NI][2];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = pf16_t{};

#pragma unroll
    for (int j = 0; j < kXReq; ++j) load_x(sb, 0, j);
#pragma unroll
    for (int j = 0; j < kWReq; ++j) load_w(sb, 0, j);
    load_s(sb);
    if (sb + 1 < se)
#pragma unroll
        for (int j = 0; j < kXReq; ++j) load_x(sb + 1, 1, j);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    store_s(0);
    zero_x(sb, 0);
    if (sb + 1 < se) zero_x(sb + 1, 1);
    __syncthreads();

    // LDS byte offsets of this lane's operands.  X: row 32 i + c of the
    // wavefront's tokens, chunk 4 g + 2 kh + h; codes: dwords 2 kh, 2 kh + 1
    // of row 64 wn + 32 j + c's group.
    const char* xl = reinterpret_cast<const char*>(Xs) + (32 * NI * wm + c) * 128;
    const char* wl = reinterpret_cast<const char*>(Ws) + (64 * wn + c) * 64 + 8 * kh;
    const char* sl = reinterpret_cast<const char*>(Ss) + (64 * wn + c) * 8;
    const int xq = 16 * ((2 * kh) ^ (c & 7)), wq = 16 * ((c >> 2) & 3);
    ph8_t af[NI][2];
    pf16_t p[2];
    uint4 w[2][2];
    uint2 cw[2];
    uint16_t sh[2];
    float sc[2];
    // tile t of a stage: group t / 2, weight rows 32 (t % 2) .. +31
    auto frag = [&](const char* x, int g, int i, int h) {
        af[i][h] = __builtin_bit_cast(ph8_t, *reinterpret_cast<const uint4*>(x + 4096 * i + (xq ^ (16 * (4 * g + h)))));
    };
    auto fetch = [&](int t, const char* wp, const char* ss, int half) {  // half: the stage of the two
        const int g = 2 * half + t / 2;
        cw[t & 1] = *reinterpret_cast<const uint2*>(wp + 2048 * (t & 1) + (wq ^ (16 * g)));
        sh[t & 1] = *reinterpret_cast<const uint16_t*>(ss + 256 * (t & 1) + 2 * g);
    };
    auto convert = [&](int t, int piece) {  // piece 0..7: pair piece % 4 of dword piece / 4
        const uint32_t d = piece < 4 ? cw[t & 1].x : cw[t & 1].y;
        const uint32_t lo = d & 0x0F0F0F0Fu, hi = (d >> 4) & 0x0F0F0F0Fu;
        uint4& o = w[t & 1][piece >> 2];
        if (piece % 4 == 0) o.x = pf_code_pair<0>(lo, hi);
        if (piece % 4 == 1) o.y = pf_code_pair<1>(lo, hi);
        if (piece % 4 == 2) o.z = pf_code_pair<2>(lo, hi);
        if (piece % 4 == 3) o.w = pf_code_pair<3>(lo, hi);
        if (piece == 7) {
            sc[t & 1] = h2f_bits(sh[t & 1]);
            asm volatile("" : "+v"(sc[t & 1]));  // converted once, not inside mixed-precision fmas at half their rate
        }
    };
    auto scale = [&](int u) {  // unit u of a stage: tile u / NI, tokens 32 (u % NI) .. +31
        const int t = u / NI, i = u % NI, j = t & 1;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = fmaf(p[u & 1][r], sc[t & 1], acc[i][j][r]);
        asm volatile("" : "+v"(acc[i][j]));  // here, not at the stage's end
    };
    p[1] = pf16_t{};
    sc[1] = 0.0f;
    fetch(0, wl, sl, 0);
    fetch(1, wl, sl, 0);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        frag(xl, 0, i, 0);
        frag(xl, 0, i, 1);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) convert(0, k);

    // Units in order; the scale fma of unit u - 1 follows the products of unit
    // u.  A stage's operands are read during the stage before, past the
    // barrier in that stage's middle, where every wavefront has seen its own
    // requests for them land; the requests then made go to buffers that every
    // wavefront has left.
    int buf = 0, wb = 0;
    auto stage = [&](auto half_c, int s) {
        constexpr int half = decltype(half_c)::value;  // of the two stages that share a code buffer
        const int nbuf = buf == 2 ? 0 : buf + 1, lbuf = nbuf == 2 ? 0 : nbuf + 1;
        const char *xc = xl + buf * (BM * 128), *xn = xl + nbuf * (BM * 128);
        const int nwb = wb ^ half;  // the next stage's code buffer
        const char *wc = wl + wb * (64 * kPfBN), *wnx = wl + nwb * (64 * kPfBN);
        const char *scu = sl + wb * (8 * kPfBN), *snx = sl + nwb * (8 * kPfBN);
        // (past the last stage its requests are made again, to buffers no
        // longer read, so that no unit holds a branch)
        const int sx = min(s + 2, se - 1), sw = s + 2 < se ? s + 2 : s;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if (t == 2) {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                if (half == 1) store_s(wb ^ 1);
                if (!FAST && s + 1 < se) zero_x(s + 1, nbuf);
                if (half == 1 || !FAST) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
            }
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const int u = t * NI + i;
                pf16_t q = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i][0], __builtin_bit_cast(ph8_t, w[t & 1][0]),
                                                                 pf16_t{}, 0, 0, 0);
                q = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i][1], __builtin_bit_cast(ph8_t, w[t & 1][1]), q, 0, 0, 0);
                p[u & 1] = q;
                __builtin_amdgcn_sched_barrier(0);
                if (t & 1) {  // the last use of this group's operands
                    frag(t == 1 ? xc : xn, t == 1 ? 1 : 0, i, 0);
                    frag(t == 1 ? xc : xn, t == 1 ? 1 : 0, i, 1);
                }
                if (i == 0)  // two tiles ahead; its code words' slot was converted during the tile before
                    fetch((t + 2) & 3, t < 2 ? wc : wnx, t < 2 ? scu : snx, t < 2 ? half : half ^ 1);
                // the requests of stage s + 2, spread over the stage's second
                // half: together they would fill the request queue and hold up
                // the products behind them
#pragma unroll
                for (int r = 0; r < kXReq + kWReq; ++r)
                    if (r * 2 * NI / (kXReq + kWReq) == u - 2 * NI) {
                        if (r < kXReq) {
                            load_x(sx, lbuf, r);
                        } else if (half == 0) {
                            load_w(sw, wb ^ 1, r - kXReq);
                            if (r == kXReq) load_s(sw);
                        }
                    }
                scale(u > 0 ? u - 1 : 4 * NI - 1);  // (the first: the last stage's last unit)
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    if (k * NI / 8 == i) convert((t + 1) & 3, k);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        buf = nbuf;
        wb = nwb;
    };
    for (int s = sb; s < se; s += 2) {
        stage(std::integral_constant<int, 0>{}, s);
        if (!FAST && s + 1 >= se) break;
        stage(std::integral_constant<int, 1>{}, s + 1);
    }
    scale(4 * NI - 1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the last requests' writes to LDS

    // tile (i, j): lane (c, kh) holds weight row n0 + 64 wn + 32 j + c for
    // tokens m0 + 32 (NI wm + i) + 8 (r / 4) + 4 kh + r % 4, r < 16; the sums
    // carry the codes' 2^-9
    auto store = [&](auto inside) {
        constexpr bool kInside = decltype(inside)::value;
        const int nb = n0 + 64 * wn + c, mb = m0 + 32 * NI * wm + 4 * kh;
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = mb + 32 * i + 8 * (r >> 2) + (r & 3);
                if (!kInside && m >= M) continue;
                float* y = nullptr;
                if (EPI == PF_PART) y = a.kpart + ((size_t)ks * M + m) * N + nb;
                else if (EPI != PF_SWIGLU) y = a.y32 + (size_t)m * a.ldy + nb;
                uint16_t* act = EPI == PF_SWIGLU ? a.act16 + (size_t)m * a.lda + (nb >> 1) : nullptr;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const float v = acc[i][j][r] * 512.0f;
                    if (EPI == PF_SWIGLU) {
                        const float u = lane_xor1(v);  // the up row n + 1 sits in lane c + 1
                        if ((c & 1) == 0 && (kInside || nb + 32 * j + 1 < N))
                            act[16 * j] = pf_swiglu(v, u);
                    } else if (kInside || nb + 32 * j < N) {
                        y[32 * j] = EPI == PF_ACC ? y[32 * j] + v : v;
                    }
                }
            }
    };
    if (m0 + BM <= M && n0 + kPfBN <= N) store(std::true_type{});
    else store(std::false_type{});
}

__global__ __launch_bounds__(256) void k_pf_embed(const int32_t* tokens, const uint16_t* embed, float* h, int d,
                                                  int vocab) {
    int tok = tokens[blockIdx.x];
    if (tok < 0 || tok >= vocab) tok = 0;  // the host checked the prompt; never index outside the table
    const uint16_t* src = embed + (size_t)tok * d;
    float* dst = h + (size_t)blockIdx.x * d;
    for (int i = threadIdx.x; i < d; i += 256) dst[i] = h2f_bits(src[i]);
}

// RoPE of the q and k rows of token t at position p0 + t (the rotation of
// the decode QKV epilogue), q to q32 [P][qdim], k and v (fp16, RNE) into
// the pages of the sequence (block table row bt).
// kvrows != nullptr (TurboQuant pages): K and V rows go there as fp32
// [P][2][kvdim] for the encoder instead of into fp16 pages.
__global__ __launch_bounds__(256) void k_pf_rope_kv(const float* qkv, int ld, int P, int p0, int qdim, int kvdim,
                                                    int hd, int hkv, const float* cos_t, const float* sin_t,
                                                    const int32_t* bt, uint16_t* kpool, uint16_t* vpool, float* q32,
                                                    float* kvrows) {
    const int npair = (qdim + 2 * kvdim) / 2;
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (long)P * npair) return;
    const int t = (int)(idx / npair), row = 2 * (int)(idx % npair), p = p0 + t, half = hd >> 1;
    float v0 = qkv[(size_t)t * ld + row], v1 = qkv[(size_t)t * ld + row + 1];
    if (row < qdim + kvdim) {
        const int i = (row % hd) >> 1;
        const float c = cos_t[(size_t)p * half + i], s = sin_t[(size_t)p * half + i];
        const float r0 = v0 * c - v1 * s;
        const float r1 = v0 * s + v1 * c;
        v0 = r0;
        v1 = r1;
    }
    if (row < qdim) {
        q32[(size_t)t * qdim + row] = v0;
        q32[(size_t)t * qdim + row + 1] = v1;
        return;
    }
    const int kv = row < qdim + kvdim ? 0 : 1, j = row - qdim - kv * kvdim, kvh = j / hd, dd = j % hd;
    if (kvrows) {
        kvrows[((size_t)t * 2 + kv) * kvdim + j] = v0;
        kvrows[((size_t)t * 2 + kv) * kvdim + j + 1] = v1;
        return;
    }
    const size_t page = ((size_t)bt[p / kPage] * hkv + kvh) * kPage * hd;
    if (kv) {  // V pages are dimension-major [hd][16]
        vpool[page + (size_t)dd * kPage + p % kPage] = f2h_bits(v0);
        vpool[page + (size_t)(dd + 1) * kPage + p % kPage] = f2h_bits(v1);
    } else {   // K pages are token-major [16][hd]
        kpool[page + (size_t)(p % kPage) * hd + dd] = f2h_bits(v0);
        kpool[page + (size_t)(p % kPage) * hd + dd + 1] = f2h_bits(v1);
    }
}

}  // namespace

namespace {

// Sum of the K parts of a split product in part order, then the epilogue.
// VEC: four columns per thread (N and the output rows multiples of 4,
// aligned); otherwise two (PF_SWIGLU: a gate/up pair) or one.
template <int EPI, bool VEC>
__global__ __launch_bounds__(256) void k_pf_ksum(PfGemmArgs a, int ksplit) {
    constexpr int C = VEC ? 4 : EPI == PF_SWIGLU ? 2 : 1;
    const size_t per = (size_t)a.M * a.N, i = ((size_t)blockIdx.x * 256 + threadIdx.x) * C;
    if (i >= per) return;
    float s[C];
#pragma unroll
    for (int c = 0; c < C; ++c) s[c] = 0.0f;
    for (int q = 0; q < ksplit; ++q) {
        const float* p = a.kpart + q * per + i;
        if constexpr (VEC) {
            const float4 v = *reinterpret_cast<const float4*>(p);
            s[0] += v.x;
            s[1] += v.y;
            s[2] += v.z;
            s[3] += v.w;
        } else {
#pragma unroll
            for (int c = 0; c < C; ++c) s[c] += p[c];
        }
    }
    const size_t m = i / a.N, n = i - m * a.N;
    if constexpr (EPI == PF_SWIGLU) {
        uint16_t* o = a.act16 + m * a.lda + (n >> 1);
#pragma unroll
        for (int c = 0; c < C; c += 2) o[c >> 1] = pf_swiglu(s[c], s[c + 1]);
    } else {
        float* y = a.y32 + m * a.ldy + n;
#pragma unroll
        for (int c = 0; c < C; ++c) y[c] = EPI == PF_ACC ? y[c] + s[c] : s[c];
    }
}

// Tile shapes (WM wavefronts along the tokens x 32 NI tokens each, 256 weight
// rows): tokens per block, blocks a CU holds, and the time of one stage (64
// k) in a block with the CU full and alone on it.  These and the constants
// below are fitted to the times of every shape and split of 320 products (M
// 16 to 2048, N 256 to 28672, K 256 to 14336): the plans chosen take 1.01
// times the best one's time in the mean, 1.14 at most.  (With one stage time
// for both: 1.03 and 1.43: 128 x 8192 x 1024 was split in four, 19.5 us, where
// one launch takes 13.7, and 200 x 4096 x 712 took 16.8 us, 13.5 now.)
struct PfShape {
    int wm, ni, occ;
    double stage_us, alone_us;
};
constexpr PfShape kPfShapes[] = {{2, 4, 1, 1.91, 1.91}, {2, 2, 1, 1.18, 1.18}, {1, 2, 2, 1.35, 0.98}, {1, 1, 2, 0.87, 0.63}};
constexpr int kPfNumShapes = 4;
constexpr int kPfMaxParts = 32, kPfMinStages = 4;  // K parts, stages of one
constexpr double kPfRoundUs = 3.0;       // a block's first round trips and its output
constexpr double kPfLaunchUs = 2.4;      // one more launch
constexpr double kPfPartUs = 0.29;       // a part's load in the sums' launch
constexpr double kPfPartBytesUs = 6.1e6; // part sums: bytes written and read per us
// An XCD's blocks walk groups of 4 token tiles; those of a last group of one
// or two share their weights with fewer others, all of them in the last XCD,
// which fetches so many bytes per us (281 x 28672 x 4096 in 32-token tiles, 9
// of them: 193 us, 119 by the stages alone; 130 in 256-token tiles).
constexpr double kPfXcdBytesUs = 3.9e5;
constexpr int kPfStageBytes = kPfBN * kPfBK * 9 / 16;  // codes and scales of a stage

struct PfPlan {
    double us = 1e30;
    int shape = 0, ksplit = 1, sper = 0;
};

// The shape and K split with the least estimated time for columns n of the
// product: rounds of blocks over the chip, plus the part sums' traffic.
// kpart_floats bounds the split.
PfPlan pf_plan(int M, int n, int G, int cus, size_t kpart_floats, bool fast) {
    const int nstage = (G + 1) / 2, ntn = (n + kPfBN - 1) / kPfBN;
    PfPlan best;
    for (int c = 0; c < kPfNumShapes; ++c) {
        const PfShape& sh = kPfShapes[c];
        if (!fast && sh.ni == 4) continue;  // (the general kernel's addresses do not fit beside this shape's sums)
        const int bm = 32 * sh.wm * sh.ni, ntm = (M + bm - 1) / bm;
        if (c + 1 < kPfNumShapes && M <= bm / 2) continue;  // half of every tile past the last token
        for (int ks = 1; ks <= kPfMaxParts; ks += ks < 8 ? 1 : 4) {
            // whole pairs of stages per part (codes are requested two stages at a time)
            const int sper = ((nstage + ks - 1) / ks + 1) / 2 * 2;
            if (ks > 1 && (sper < kPfMinStages || (size_t)ks * M * n > kpart_floats || (nstage + sper - 1) / sper != ks)) continue;
            const long blocks = (long)ntm * ntn * ks, slots = (long)cus * sh.occ, rest = blocks % slots;
            double us = (double)(blocks / slots) * (sper * sh.stage_us + kPfRoundUs);
            if (rest > 0) us += sper * (rest <= cus ? sh.alone_us : sh.stage_us) + kPfRoundUs;
            if (ks == 1 && blocks > slots && ntm % 4 > 0) {
                const int per_xcd = cus / kPfXcds * sh.occ, g = ntm % 4;
                const long share = (blocks + kPfXcds - 1) / kPfXcds, last = std::min<long>(share, (long)ntn * g);
                const double slow = std::max(sh.stage_us, (double)std::min<long>(per_xcd, last) / g * kPfStageBytes / kPfXcdBytesUs);
                const long all = (share + per_xcd - 1) / per_xcd, end = (last + per_xcd - 1) / per_xcd;
                us = std::max(us, (all - end) * (sper * sh.stage_us + kPfRoundUs) + end * (sper * slow + kPfRoundUs));
            }
            if (ks > 1) us += kPfLaunchUs + ks * kPfPartUs + 8.0 * ks * M * n / kPfPartBytesUs;
            if (us < best.us) best = {us, c, ks, sper};
        }
    }
    return best;
}

// Columns [0, cut) and [cut, N) as two launches where the first fills whole
// rounds of the chip with the tiles of one shape and the rest, which would be
// a partial round of them, takes another (M 2048, N 28672, K 4096: 3.5 rounds
// of 256 x 256 tiles; 540 us in four rounds).  Every shape's cut is weighed
// against the best single launch (1481 x 11008 x 4096: 161 us in two launches,
// 232 in the 32-token tiles that are the best alone).
// cut = N: one launch.
int pf_cut(int M, int N, int G, int cus, size_t kpart_floats, bool fast, PfPlan& first, PfPlan& rest) {
    first = pf_plan(M, N, G, cus, kpart_floats, fast);
    if (!fast || first.ksplit > 1) return N;
    const int ntn = (N + kPfBN - 1) / kPfBN, sper = ((G + 1) / 2 + 1) / 2 * 2;
    int cut = N;
    for (int c = 0; c < kPfNumShapes; ++c) {
        const PfShape& sh = kPfShapes[c];
        const int bm = 32 * sh.wm * sh.ni, ntm = (M + bm - 1) / bm, slots = cus * sh.occ;
        if (c + 1 < kPfNumShapes && M <= bm / 2) continue;
        const int cols = (int)((long)ntm * ntn / slots * slots / ntm);
        if (cols < 1 || cols >= ntn) continue;
        const long rounds = ((long)ntm * cols + slots - 1) / slots;
        const double whole = rounds * (sper * sh.stage_us + kPfRoundUs) + kPfLaunchUs;
        if (whole >= first.us) continue;
        const PfPlan r = pf_plan(M, N - cols * kPfBN, G, cus, kpart_floats, fast);
        if (whole + r.us >= first.us) continue;
        first = {whole + r.us, c, 1, sper};
        rest = r;
        cut = cols * kPfBN;
    }
    return cut;
}

bool pf_fast(const PfGemmArgs& a) {
    return a.K % 128 == 0 && (reinterpret_cast<uintptr_t>(a.S) & 7u) == 0 && a.ldx < (1 << 22) && a.G < (1 << 18);
}

hipError_t pf_gemm_part(int epi, const PfGemmArgs& a, const PfPlan& pl, bool fast, hipStream_t st) {
    const PfShape& sh = kPfShapes[pl.shape];
    const int bm = 32 * sh.wm * sh.ni;
    PfTiles tl;
    tl.ntm = (a.M + bm - 1) / bm;
    tl.ntn = (a.N + kPfBN - 1) / kPfBN;
    tl.ksplit = pl.ksplit;
    tl.sper = pl.sper;
    const long T = (long)tl.ntm * tl.ntn * tl.ksplit;
    if (T > 0x3FFFFFFFL) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((T + kPfXcds - 1) / kPfXcds * kPfXcds));
    const int e = pl.ksplit > 1 ? (int)PF_PART : epi;
#define NX_PF_SHAPE(E, C)                                                                                          \
    case C:                                                                                                        \
        if constexpr (kPfShapes[C].ni < 4)                                                                         \
            if (!fast) {                                                                                           \
                hipLaunchKernelGGL((k_pf_gemm<E, kPfShapes[C].wm, kPfShapes[C].ni, false>), grid,                  \
                                   dim3(kPfThreads * kPfShapes[C].wm), 0, st, a, tl);                              \
                break;                                                                                             \
            }                                                                                                      \
        hipLaunchKernelGGL((k_pf_gemm<E, kPfShapes[C].wm, kPfShapes[C].ni, true>), grid,                           \
                           dim3(kPfThreads * kPfShapes[C].wm), 0, st, a, tl);                                      \
        break;
#define NX_PF_CASE(E)                                                                                              \
    case E:                                                                                                        \
        switch (pl.shape) { NX_PF_SHAPE(E, 0) NX_PF_SHAPE(E, 1) NX_PF_SHAPE(E, 2) NX_PF_SHAPE(E, 3) }              \
        break;
    switch (e) {
        NX_PF_CASE(PF_F32)
        NX_PF_CASE(PF_ACC)
        NX_PF_CASE(PF_SWIGLU)
        NX_PF_CASE(PF_PART)
        default: return hipErrorInvalidValue;
    }
#undef NX_PF_CASE
#undef NX_PF_SHAPE
    hipError_t err = hipGetLastError();
    if (err != hipSuccess || pl.ksplit == 1) return err;
    const bool vec = a.N % 4 == 0 && (epi == PF_SWIGLU || (a.ldy % 4 == 0 && (reinterpret_cast<uintptr_t>(a.y32) & 15u) == 0)) &&
                     (reinterpret_cast<uintptr_t>(a.kpart) & 15u) == 0;
    const size_t items = (size_t)a.M * a.N / (vec ? 4 : epi == PF_SWIGLU ? 2 : 1);
    const dim3 g2((unsigned)((items + 255) / 256));
#define NX_PF_SUM(E)                                                                                  \
    case E:                                                                                           \
        if (vec) hipLaunchKernelGGL((k_pf_ksum<E, true>), g2, dim3(256), 0, st, a, pl.ksplit);        \
        else hipLaunchKernelGGL((k_pf_ksum<E, false>), g2, dim3(256), 0, st, a, pl.ksplit);           \
        break;
    switch (epi) {
        NX_PF_SUM(PF_F32)
        NX_PF_SUM(PF_ACC)
        NX_PF_SUM(PF_SWIGLU)
    }
#undef NX_PF_SUM
    return hipGetLastError();
}

}  // namespace

size_t pf_gemm_part_floats(int M, int N, int K) {
    const int G = (K + 31) / 32, cus = device_cus();
    PfPlan p, r;
    const int cut = pf_cut(M, N, G, cus, kPfPartMaxFloats, K % 128 == 0, p, r);
    size_t need = p.ksplit > 1 ? (size_t)p.ksplit * M * N : 0;
    if (cut < N && r.ksplit > 1) need = std::max(need, (size_t)r.ksplit * M * (N - cut));
    return need;
}

size_t pf_gemm_part_bound(int M, int N, int K) {
    const int stages = (K + kPfBK - 1) / kPfBK;
    return std::min(kPfPartMaxFloats, (size_t)std::min(kPfMaxParts, (stages + 3) / kPfMinStages) * M * N);
}

size_t pf_gemm_part_floats_upto(int M, int N, int K) {
    size_t most = 0;
    for (int m = 1; m <= M; ++m) most = std::max(most, pf_gemm_part_floats(m, N, K));
    return most;
}

hipError_t pf_gemm_launch(int epi, const PfGemmArgs& a, hipStream_t st) {
    // 16-byte rows of x (K and ldx multiples of 8, aligned base), at least one
    // full 8-k chunk
    if (a.M < 1 || a.N < 1 || a.K < 8 || a.K % 8 || a.ldx % 8 || (reinterpret_cast<uintptr_t>(a.x) & 15) ||
        a.G != (a.K + 31) / 32 || (epi == PF_SWIGLU && a.N % 2) || epi < PF_F32 || epi > PF_SWIGLU)
        return hipErrorInvalidValue;
    const bool fast = pf_fast(a);
    PfPlan p, r;
    const int cut = pf_cut(a.M, a.N, a.G, device_cus(), a.kpart ? a.kpart_floats : 0, fast, p, r);
    if (cut == a.N) return pf_gemm_part(epi, a, p, fast, st);
    PfGemmArgs f = a, g = a;
    f.N = cut;
    g.N = a.N - cut;
    g.W = a.W + (size_t)cut * a.G * 16;
    g.S = a.S + (size_t)cut * a.G;
    if (a.y32) g.y32 = a.y32 + cut;
    if (a.act16) g.act16 = a.act16 + cut / 2;
    const hipError_t e = pf_gemm_part(epi, f, p, fast, st);
    return e != hipSuccess ? e : pf_gemm_part(epi, g, r, fast, st);
}

hipError_t pf_embed_launch(const int32_t* tokens, int P, const uint16_t* embed, float* h, int d, int vocab,
                           hipStream_t st) {
    hipLaunchKernelGGL(k_pf_embed, dim3(P), dim3(256), 0, st, tokens, embed, h, d, vocab);
    return hipGetLastError();
}

hipError_t pf_rope_kv_launch(const float* qkv, int ld, int P, int p0, int qdim, int kvdim, int hd, int hkv,
                             const float* cos_t, const float* sin_t, const int32_t* bt, uint16_t* kpool,
                             uint16_t* vpool, float* q32, hipStream_t st, float* kvrows) {
    const long n = (long)P * ((qdim + 2 * kvdim) / 2);
    hipLaunchKernelGGL(k_pf_rope_kv, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, qkv, ld, P, p0, qdim, kvdim,
                       hd, hkv, cos_t, sin_t, bt, kpool, vpool, q32, kvrows);
    return hipGetLastError();
}

}  // namespace nx
