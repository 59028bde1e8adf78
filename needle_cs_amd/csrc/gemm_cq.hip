// gemm_cq.hip -- prefill matmul of the codebook formats (many tokens) on
// gfx950.
//
// y[t][n] for a block of 16 * TI tokens x 64 * TPW weight rows per workgroup:
// each of the four waves owns TPW 16-row weight tiles and all the tokens, so a
// tile's codes go through the codebook once for 16 * TI tokens and its
// activations are read once for four waves (gemv.hip's general kernel does
// both for every 16 x 16 block).  Per 128-element group two
// v_mfma_i32_16x16x64_i8 per (16-token subtile, tile) give the exact int32
// D_g; lane l then holds D_g for row l%16 and tokens 4*(l/16)..+3 of the
// subtile and runs Scalar.MatMulRows' chain (Scalar.cs:159-189) over the groups
// in ascending order in its registers:
//   scaled = (h(norm[n][g]) * ByteScale) * scale[t][g]
//   acc += scaled * D_g ;  bias += scaled * offset[t][g] ;  y = acc - bias
//
// What bounds it: on large grids the VALU -- the chain's six operations per
// (token, row, group) and the lookups and addresses, about 60 per (tile, group)
// of a wave; counters show it issuing in 73% of the cycles, the MFMAs in 13%.
// On small ones the length of a wave's chain over the groups, about 0.4 us a
// group.  Measured, one launch among others (general kernel before):
//   Cq4  512 x 2048 x 8192    29.4 us (90.9)     64 x 128 tile
//   Cq2 1024 x 2048 x 4096    28.2 us (139.5)    64 x 128
//   Cq4  256 x 2048 x 4096    13.5 us (25.8)     32 x 64
//   Cq2   61 x  768 x 1568     4.3 us (10.5)     16 x 64
// A 128 x 64 tile halves the lookups per token but not the time (33.8 us for
// the first shape: twice the LDS reads per MFMA); one wave per 16 x 16 tile
// with operands straight from memory took 5.1 us for the last.
//
// Activations go through LDS, two groups a stage, copied straight from memory
// (global_load_lds, no registers) and double-buffered; the groups' scales and
// offsets beside them, [group][token], so that a lane reads its four tokens in
// one ds_read_b128.  Weight blocks and norms stream one stage ahead in
// registers.
#include <algorithm>

#include "common.hpp"

namespace nhip {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));

constexpr int kWaitVmcnt0 = 0x0F70;  // s_waitcnt: vmcnt 0 only
constexpr int kGroups = 2;           // groups per stage (4 and 8 measured no faster)
// LDS bytes of a stage of 16 * TI tokens: the activations, and the scales and
// offsets of 64 tokens (a wave's copy; past the block's own, unused)
constexpr int act_lds(int ti) { return kGroups * 128 * 16 * ti; }
constexpr int kScaleLds = kGroups * 2 * 64 * 4;
constexpr int stage_lds(int ti) { return act_lds(ti) + kScaleLds; }

template <bool CQ4, int TPW>
struct WStage {
    u4 w[CQ4 ? kGroups : kGroups / 2][TPW];
    uint32_t h[TPW][kGroups / 2];  // the stage's norms of the lane's row
};

template <bool CQ4, bool SPECIAL, int TI, int TPW>
__device__ __forceinline__ void gemm_cq_body(const TileMatmul& p)
{
    constexpr int kTokens = 16 * TI;  // per workgroup
    static_assert(TI <= 4, "a wave copies the scales of at most 64 tokens");
    __shared__ __align__(16) uint8_t lds[2 * stage_lds(TI)];
    auto alds = [&](int buf) { return lds + buf * stage_lds(TI); };
    // [group][scale / offset][token]
    auto slds = [&](int buf, int g, int o) {
        return reinterpret_cast<float*>(lds + buf * stage_lds(TI) + act_lds(TI)) + (g * 2 + o) * 64;
    };
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15;
    const int kq = lane >> 4;
    const int t0 = blockIdx.y * kTokens;
    const int G = p.groups;
    const int stages = (G + kGroups - 1) / kGroups;

    // the wave's tiles; past the last one it repeats that tile, unstored
    const int u0 = (blockIdx.x * 4 + wave) * TPW;
    const int units = p.first[p.count];
    int job[TPW], tile[TPW];
    const u4* wbase[TPW];
    const uint16_t* nrow[TPW];
    float bs[TPW];
    uint32_t tb[TPW][4];
#pragma unroll
    for (int j = 0; j < TPW; j++) {
        const int u = min(u0 + j, units - 1);
        job[j] = 0;
#pragma unroll
        for (int k = 1; k < kMaxTileJobs; k++)
            if (k < p.count && u >= p.first[k]) job[j] = k;
        const TileJob& jb = p.job[job[j]];
        tile[j] = jb.tile_begin + u - p.first[job[j]];
        wbase[j] = reinterpret_cast<const u4*>(jb.tiles) + (size_t)tile[j] * p.blocks * 64 + lane;
        nrow[j] = jb.norms + (size_t)(tile[j] * 16 + r) * p.groups_pad8;
        bs[j] = jb.byte_scale;
#pragma unroll
        for (int k = 0; k < 4; k++) tb[j][k] = jb.table[k];
    }

    // Activation staging: 4 * TI wave instructions of 1 KB a stage, TI a wave,
    // lane l's 16 bytes at 16 * l.
    //   Cq4: one (group, subtile i, slot s) each, in the MFMA's lane order: the
    //   A operand (token 16i + r, 16 bytes at 32s + 64(kq/2) + 16(kq%2) of the
    //   group) is the lane's own 16 bytes back, a conflict-free ds_read_b128.
    //   Cq2: two (plane, subtile) blocks of 512 bytes each, where position x
    //   holds the 16 bytes of token x/2 and half (x & 1) ^ bit 3 of the token
    //   of the plane's 32 (the swizzle keeps a half-wave's ds_read_b64 on
    //   different banks).
    auto load_a = [&](int buf, int st) {
#pragma unroll
        for (int j = 0; j < TI; j++) {
            const int R = TI * wave + j;
            const int8_t* src;
            if constexpr (CQ4) {
                const int g = min(st * kGroups + R / (2 * TI), G - 1), i = (R >> 1) % TI, s = R & 1;
                const int t = min(t0 + 16 * i + r, p.tokens - 1);
                src = p.q + (size_t)t * p.cols + g * 128 + 32 * s + 64 * (kq >> 1) + 16 * (kq & 1);
            } else {
                // block b = (group, plane, subtile) = (4 * group + plane) * TI + i
                const int b = 2 * R + (lane >> 5), x = lane & 31, rr = x >> 1;
                const int g = min(st * kGroups + b / (4 * TI), G - 1), pl = (b / TI) & 3, i = b % TI;
                const int t = min(t0 + 16 * i + rr, p.tokens - 1);
                src = p.q + (size_t)t * p.cols + g * 128 + 32 * pl + 16 * ((x & 1) ^ ((rr >> 3) & 1));
            }
            __builtin_amdgcn_global_load_lds(src, alds(buf) + R * 1024, 16, 0, 0);
        }
        // wave w: the scales (w even) or offsets of group w / 2, one token a lane
        const int g = min(st * kGroups + (wave >> 1), G - 1);
        const float* sc = (wave & 1) ? p.offsets : p.scales;
        __builtin_amdgcn_global_load_lds(sc + (size_t)min(t0 + lane, p.tokens - 1) * p.stride + g,
                                         slds(buf, wave >> 1, wave & 1), 4, 0, 0);
    };
    auto load_w = [&](WStage<CQ4, TPW>& x, int st) {
#pragma unroll
        for (int j = 0; j < TPW; j++) {
            constexpr int NB = CQ4 ? kGroups : kGroups / 2;  // weight blocks of a stage
#pragma unroll
            for (int b = 0; b < NB; b++) x.w[b][j] = wbase[j][(size_t)min(st * NB + b, p.blocks - 1) * 64];
            // (norm rows are padded to 8 halves)
            const uint32_t* h = reinterpret_cast<const uint32_t*>(nrow[j] + st * kGroups);
#pragma unroll
            for (int k = 0; k < kGroups / 2; k++) x.h[j][k] = h[k];
        }
    };

    float acc[TPW][TI][4], bias[TPW][TI][4];
#pragma unroll
    for (int j = 0; j < TPW; j++)
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) acc[j][i][e] = bias[j][i][e] = 0.0f;

    auto group = [&](const WStage<CQ4, TPW>& x, int buf, int k) {
        // the A operands of the TI subtiles
        v4i a[TI][2];
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int s = 0; s < 2; s++) {
                if constexpr (CQ4) {
                    a[i][s] = *reinterpret_cast<const v4i*>(alds(buf) + ((k * TI + i) * 2 + s) * 1024 + lane * 16);
                } else {
                    const int pos = (2 * r + ((kq >> 1) ^ ((r >> 3) & 1))) * 16 + (kq & 1) * 8;
                    const uint2 lo = *reinterpret_cast<const uint2*>(alds(buf) + ((k * 4 + 2 * s) * TI + i) * 512 + pos);
                    const uint2 hi = *reinterpret_cast<const uint2*>(alds(buf) + ((k * 4 + 2 * s + 1) * TI + i) * 512 + pos);
                    a[i][s] = v4i{(int)lo.x, (int)lo.y, (int)hi.x, (int)hi.y};
                }
            }
        float4 s4[TI], o4[TI];
#pragma unroll
        for (int i = 0; i < TI; i++) {
            s4[i] = *reinterpret_cast<const float4*>(slds(buf, k, 0) + 16 * i + 4 * kq);
            o4[i] = *reinterpret_cast<const float4*>(slds(buf, k, 1) + 16 * i + 4 * kq);
        }
        v4i d[TPW][TI];
#pragma unroll
        for (int j = 0; j < TPW; j++) {
            v4i b[2];
#pragma unroll
            for (int s = 0; s < 2; s++) {
                if constexpr (CQ4) {
                    const u4& wc = x.w[k][j];
                    b[s].x = (int)lut4x((wc.x >> (4 * s)) & 0x0F0F0F0Fu, tb[j][0], tb[j][1], tb[j][2], tb[j][3]);
                    b[s].y = (int)lut4x((wc.y >> (4 * s)) & 0x0F0F0F0Fu, tb[j][0], tb[j][1], tb[j][2], tb[j][3]);
                    b[s].z = (int)lut4x((wc.z >> (4 * s)) & 0x0F0F0F0Fu, tb[j][0], tb[j][1], tb[j][2], tb[j][3]);
                    b[s].w = (int)lut4x((wc.w >> (4 * s)) & 0x0F0F0F0Fu, tb[j][0], tb[j][1], tb[j][2], tb[j][3]);
                } else {  // planes 2s and 2s + 1
                    const u4& wc = x.w[k >> 1][j];
                    const uint32_t x0 = (k & 1) ? wc.z : wc.x, x1 = (k & 1) ? wc.w : wc.y;
                    b[s].x = (int)lut2((x0 >> (4 * s)) & 0x03030303u, tb[j][0]);
                    b[s].y = (int)lut2((x1 >> (4 * s)) & 0x03030303u, tb[j][0]);
                    b[s].z = (int)lut2((x0 >> (4 * s + 2)) & 0x03030303u, tb[j][0]);
                    b[s].w = (int)lut2((x1 >> (4 * s + 2)) & 0x03030303u, tb[j][0]);
                }
            }
            const v4i zero = {0, 0, 0, 0};
#pragma unroll
            for (int i = 0; i < TI; i++) d[j][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i][0], b[0], zero, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < TI; i++) d[j][i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i][1], b[1], d[j][i], 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < TPW; j++) {
            const uint32_t hbits = (k & 1) ? (x.h[j][k >> 1] >> 16) : (x.h[j][k >> 1] & 0xFFFFu);
            float hs;
            if constexpr (SPECIAL)
                hs = ref_half_to_single(hbits) * bs[j];
            else  // exact; a -0 norm adds zeros, which leave the sums as they are
                hs = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(hbits))) * bs[j];
#pragma unroll
            for (int i = 0; i < TI; i++) {
                const float sv[4] = {s4[i].x, s4[i].y, s4[i].z, s4[i].w}, ov[4] = {o4[i].x, o4[i].y, o4[i].z, o4[i].w};
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float scaled = hs * sv[e];
                    acc[j][i][e] = acc[j][i][e] + scaled * static_cast<float>(d[j][i][e]);
                    bias[j][i][e] = bias[j][i][e] + scaled * ov[e];
                }
            }
        }
    };

    // stage st + 1's loads are in flight while stage st is multiplied (the
    // last iteration reloads the last stage, unused)
    WStage<CQ4, TPW> wcur, wnext;
    load_a(0, 0);
    load_w(wcur, 0);
    __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
    __syncthreads();
    for (int st = 0; st < stages; st++) {
        const int buf = st & 1;
        const int nst = min(st + 1, stages - 1);
        load_a(buf ^ 1, nst);  // that buffer was last read before the previous barrier
        load_w(wnext, nst);
#pragma unroll
        for (int k = 0; k < kGroups; k++)
            if (k == 0 || st * kGroups + k < G) group(wcur, buf, k);
        wcur = wnext;
        __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);  // this wave's LDS copies of the next stage have landed
        __syncthreads();
    }

#pragma unroll
    for (int j = 0; j < TPW; j++) {
        const TileJob& jb = p.job[job[j]];
        const int n = tile[j] * 16 + r;
        if (u0 + j >= units || n < jb.row_start || n >= jb.row_end) continue;
        float* out = jb.y + (n - jb.row0);
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int t = t0 + 16 * i + 4 * kq + e;
                if (t < p.tokens) out[(size_t)t * jb.ldy] = acc[j][i][e] - bias[j][i][e];
            }
    }
}

template <bool CQ4, bool SPECIAL, int TI, int TPW>
__global__ __launch_bounds__(256) void gemm_cq_kernel(TileMatmul p)
{
    gemm_cq_body<CQ4, SPECIAL, TI, TPW>(p);
}

template <bool CQ4, bool SPECIAL, int TI, int TPW>
int32_t launch(const TileMatmul& p, hipStream_t s)
{
    const int tiles = p.first[p.count];
    const dim3 grid((tiles + 4 * TPW - 1) / (4 * TPW), (p.tokens + 16 * TI - 1) / (16 * TI));
    hipLaunchKernelGGL((gemm_cq_kernel<CQ4, SPECIAL, TI, TPW>), grid, dim3(256), 0, s, p);
    NHIP_CHECK_HIP(hipGetLastError());
    return NHIP_OK;
}

template <bool CQ4, int TI, int TPW>
int32_t launch(const TileMatmul& p, bool special, hipStream_t s)
{
    return special ? launch<CQ4, true, TI, TPW>(p, s) : launch<CQ4, false, TI, TPW>(p, s);
}

template <bool CQ4>
int32_t launch_form(const TileMatmul& p, bool special, hipStream_t s)
{
    const int tiles = p.first[p.count];
    const auto groups_of = [&](int ti, int tpw) {  // workgroups of a launch
        return (int64_t)((tiles + 4 * tpw - 1) / (4 * tpw)) * ((p.tokens + 16 * ti - 1) / (16 * ti));
    };
    // The largest tile whose grid gives three quarters of the 256 CUs a workgroup
    // (64 x 128), or one and a half to each (32 x 64).  64 x 128
    // takes about as long for 128 workgroups as for 256 (19.5 us at K 2048) and
    // loses to four times as many of 32 x 64 at 128 (13.5 us); 32 x 64 and
    // 16 x 64 meet near 400 (Cq2 512 x 768 x 1568, 400: 6.7 against 6.8 us;
    // 300 tokens, 250: 5.7 against 5.0 us).
    if (groups_of(4, 2) >= 192) return launch<CQ4, 4, 2>(p, special, s);
    if (groups_of(2, 1) >= 384) return launch<CQ4, 2, 1>(p, special, s);
    return launch<CQ4, 1, 1>(p, special, s);
}

}  // namespace

int32_t launch_gemm_cq(WeightFormat fmt, const TileMatmul& p, bool special, hipStream_t stream)
{
    return fmt == WeightFormat::Cq4 ? launch_form<true>(p, special, stream) : launch_form<false>(p, special, stream);
}

}  // namespace nhip
