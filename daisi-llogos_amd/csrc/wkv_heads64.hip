// The recurrence with a matrix state per head (see sequence_state.hip for what it computes) for heads of 64
// channels, the size the models use: a wave owns a head of a sequence, its whole state in registers.
//
// Lane l = 8 b + a keeps the block of S with key channels 8 a .. 8 a + 7 and value channels 8 b .. 8 b + 7, 64
// registers.  A token then costs a lane eight reads of 16 bytes from LDS (its 8 values each of r, k, the decay and v;
// a column a lane would read 48, three times what the LDS serves beside the arithmetic), 192 multiply-adds and 22
// instructions that add the eight lanes' sums of a value channel and leave channel l with lane l, where the head's
// norm, the gate and the store are one channel a lane.  What bounds it is those instructions: the plain multiply-adds
// of a token and head are 192 x 4 clocks.  The bonus enters as (sum_i r_i u_i k_i) v_j, eight products a lane instead
// of one for every element of S.
// Tokens come in chunks of 8: a chunk's values are asked for (a channel a lane, whole lines) while the one before is
// worked on.  Waves do not share anything, so nothing waits at a barrier.
// Long prompts are cut into segments as in sequence_state.hip (MODE 1: end state from zero and the product of the
// decays; wkv_combine; MODE 2: the outputs from the true initial state); a token's arithmetic is the same in all modes.
// Measured (us, 64 heads, before in the kernel of sequence_state.hip -> now): eight prompts of 250 to 600 tokens 864 -> 281,
// one of 2,048 454 -> 158, one of 8,000 1,449 -> 535; single tokens of 64 sequences 114 -> 26.
#include "common.h"

#pragma clang fp contract(off)      // (the same roundings whatever a form's surroundings let the compiler fuse)

constexpr int kWkvDim = 64, kWkvWaves = 4;

template <int CTRL>
__device__ __forceinline__ float wkv_dpp(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false));
}
// x of lane l ^ 4: lanes of the even groups of four read four lanes further, the others four lanes back
__device__ __forceinline__ float wkv_xor4(float x) {
    const int v = __float_as_int(x);
    int o = __builtin_amdgcn_update_dpp(0, v, 0x104, 0xf, 0x5, false);           // row_shl:4
    o = __builtin_amdgcn_update_dpp(o, v, 0x114, 0xf, 0xa, false);               // row_shr:4
    return __int_as_float(o);
}
// the sums over the eight lanes of a group of eight values each; lane a of the group gets value a's
__device__ __forceinline__ float wkv_sum8(const float (&p)[8], int lane) {
    float q[4], s[2];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float keep = lane & 1 ? p[2 * e + 1] : p[2 * e], give = lane & 1 ? p[2 * e] : p[2 * e + 1];
        q[e] = keep + wkv_dpp<0xB1>(give);                                       // quad_perm: lane ^ 1
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const float keep = lane & 2 ? q[2 * e + 1] : q[2 * e], give = lane & 2 ? q[2 * e] : q[2 * e + 1];
        s[e] = keep + wkv_dpp<0x4E>(give);                                       // quad_perm: lane ^ 2
    }
    const float keep = lane & 4 ? s[1] : s[0], give = lane & 4 ? s[0] : s[1];
    return keep + wkv_xor4(give);
}

// C: tokens a chunk, 8, or 1 for single-token steps
template <int MODE, int C, typename TO>
__global__ __launch_bounds__(kWkvWaves * kWave) void wkv64_kernel(
        TO* __restrict__ y, const float* __restrict__ r, const float* __restrict__ k, const float* __restrict__ v,
        const float* __restrict__ d, const float* __restrict__ gate, int ld, int parts, size_t part_stride, int d_parts,
        size_t d_part_stride, const float* __restrict__ w0, const float* __restrict__ u, const float* __restrict__ g, float eps,
        float* __restrict__ state, size_t state_stride, size_t prev_offset, const float* __restrict__ h_in, int W,
        const int* __restrict__ slots, const int* __restrict__ cu, int H, int n_seg, int seg_len,
        float* __restrict__ seg_state, float* __restrict__ seg_decay) {
    constexpr int D = kWkvDim;
    __shared__ __align__(16) float lds[kWkvWaves][4][C * D];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, a = lane & 7, b = lane >> 3;
    const int head = blockIdx.x * kWkvWaves + wave, seq = blockIdx.y, seg = blockIdx.z;
    const int first0 = cu ? cu[seq] : seq, count0 = cu ? cu[seq + 1] - first0 : 1;
    float* row = state + (size_t)slots[seq] * state_stride;
    // the step's last mixer input row becomes the sequence's `prev` row (the token shift has read the old one by then)
    if (MODE != 1 && seg == 0 && h_in && count0 > 0) {
        const float* last = h_in + (size_t)(first0 + count0 - 1) * W;
        for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < W; c += gridDim.x * blockDim.x) row[prev_offset + c] = last[c];
    }
    if (head >= H) return;
    const int first = first0 + (MODE ? seg * seg_len : 0);
    const int count = MODE ? min(seg_len, count0 - seg * seg_len) : count0;
    const size_t at = ((size_t)seq * n_seg + seg) * H + head;
    float* S = MODE ? seg_state + at * D * D : row + (size_t)head * D * D;      // [value channel][key channel]
    if (count <= 0) {                                       // (in mode 0 a sequence that brings no token: its state stays)
        if (MODE == 1) {                                    // a segment beyond the sequence's end: nothing added, nothing decayed
            for (int e = lane; e < D * D; e += kWave) S[e] = 0.f;
            seg_decay[at * D + lane] = 1.f;
        }
        return;
    }
    const int col = head * D + lane;                        // this lane's channel where a lane is a channel
    float s[8][8], ur[8], pw[8];                            // s[value channel][key channel]
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int i = 0; i < 8; i += 4) {
            const float4 q = MODE == 1 ? make_float4(0.f, 0.f, 0.f, 0.f) : *reinterpret_cast<const float4*>(S + (8 * b + j) * D + 8 * a + i);
            s[j][i] = q.x; s[j][i + 1] = q.y; s[j][i + 2] = q.z; s[j][i + 3] = q.w;
        }
#pragma unroll
    for (int i = 0; i < 8; ++i) { ur[i] = u[head * D + 8 * a + i]; pw[i] = 1.f; }
    const float decay0 = w0[col], gain = MODE == 1 ? 0.f : g[col];

    float pr[C], pk[C], pv[C], pd[C], pg[C], gz[C];
    auto ask = [&](int c0) {
        const int n = min(C, count - c0);
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const size_t p = (size_t)(first + c0 + min(c, n - 1)) * ld + col;
            pk[c] = k[p]; pv[c] = v[p]; pd[c] = d[p];
            if (MODE != 1) { pr[c] = r[p]; pg[c] = gate[p]; }
        }
        for (int q = 1; q < parts; ++q)                     // products that come as partial sums of a split along k
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const size_t p = q * part_stride + (size_t)(first + c0 + min(c, n - 1)) * ld + col;
                pk[c] += k[p]; pv[c] += v[p];
                if (MODE != 1) { pr[c] += r[p]; pg[c] += gate[p]; }
            }
        for (int q = 1; q < d_parts; ++q)
#pragma unroll
            for (int c = 0; c < C; ++c) pd[c] += d[q * d_part_stride + (size_t)(first + c0 + min(c, n - 1)) * ld + col];
    };
    float (&sr)[C * D] = lds[wave][0], (&sk)[C * D] = lds[wave][1], (&sw)[C * D] = lds[wave][2], (&sv)[C * D] = lds[wave][3];
    ask(0);
    for (int c0 = 0; c0 < count; c0 += C) {
        const int n = min(C, count - c0);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int c = 0; c < C; ++c) {
            if (MODE != 1) { sr[c * D + lane] = pr[c]; gz[c] = pg[c]; }
            // (behind the last token: a token that adds nothing and lets nothing decay, so that the loop has no branch)
            sk[c * D + lane] = c < n ? pk[c] : 0.f;
            sv[c * D + lane] = c < n ? pv[c] : 0.f;
            sw[c * D + lane] = c < n ? expf(-expf(pd[c] + decay0)) : 1.f;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");      // (a wave's LDS operations run in order)
        if (c0 + C < count) ask(c0 + C);
        float o[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            float rv[8], kv[8], wv[8], vv[8], part[8];
            auto read8 = [&](float (&x)[8], const float* p) {
                const float4 lo = *reinterpret_cast<const float4*>(p), hi = *reinterpret_cast<const float4*>(p + 4);
                x[0] = lo.x; x[1] = lo.y; x[2] = lo.z; x[3] = lo.w; x[4] = hi.x; x[5] = hi.y; x[6] = hi.z; x[7] = hi.w;
            };
            read8(kv, sk + c * D + 8 * a);
            read8(wv, sw + c * D + 8 * a);
            read8(vv, sv + c * D + 8 * b);
            if (MODE != 1) {
                read8(rv, sr + c * D + 8 * a);
                float bonus = 0.f;
#pragma unroll
                for (int i = 0; i < 8; ++i) bonus = fmaf(rv[i] * ur[i], kv[i], bonus);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    float x = bonus * vv[j];
#pragma unroll
                    for (int i = 0; i < 8; ++i) x = fmaf(rv[i], s[j][i], x);
                    part[j] = x;
                }
                o[c] = wkv_sum8(part, lane);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int i = 0; i < 8; ++i) s[j][i] = fmaf(wv[i], s[j][i], kv[i] * vv[j]);
            if (MODE == 1) {
#pragma unroll
                for (int i = 0; i < 8; ++i) pw[i] *= wv[i];
            }
        }
        if (MODE == 1) continue;
        // the head's norm, for the eight tokens of a chunk at once: lane c of a group of eight sums token c
        float ss;
        if (C == 8) {
            float sq[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) sq[c] = o[c % C] * o[c % C];
            ss = wkv_sum8(sq, lane);
        } else {
            ss = o[0] * o[0];
            ss += wkv_dpp<0xB1>(ss);
            ss += wkv_dpp<0x4E>(ss);
            ss += wkv_xor4(ss);
        }
        ss += wkv_dpp<0x128>(ss);                                               // row_ror:8, the other group of the row of 16
        ss += __shfl_xor(ss, 16, kWave);
        ss += __shfl_xor(ss, 32, kWave);
        const float inv = 1.0f / sqrtf(ss / (float)D + eps);
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const float scale = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(inv), c));
            if (c < n) store_f32(y + (size_t)(first + c0 + c) * H * D + col, o[c] * scale * gain * (gz[c] / (1.0f + expf(-gz[c]))));
        }
    }
    if (MODE != 2) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int i = 0; i < 8; i += 4)
                *reinterpret_cast<float4*>(S + (8 * b + j) * D + 8 * a + i) = make_float4(s[j][i], s[j][i + 1], s[j][i + 2], s[j][i + 3]);
    }
    if (MODE == 1 && b == 0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) seg_decay[at * D + 8 * a + i] = pw[i];
    }
}

// The segments' local end states chained: seg_state[seg] <- the state the segment starts from, and the cached state <- the
// state after the last segment.  A thread owns four key channels of one value channel.
__global__ __launch_bounds__(256) void wkv64_combine_kernel(float* __restrict__ state, size_t state_stride, const int* __restrict__ slots,
                                                            float* __restrict__ seg_state, const float* __restrict__ seg_decay, int H, int n_seg) {
    constexpr int D = kWkvDim;
    const int head = blockIdx.x, seq = blockIdx.y, e = (blockIdx.z * 256 + threadIdx.x) * 4, i = e % D;
    float4* S = reinterpret_cast<float4*>(state + (size_t)slots[seq] * state_stride + (size_t)head * D * D + e);
    float4 cur = *S;
    const size_t at = (size_t)seq * n_seg * H + head;
    float4 local = *reinterpret_cast<const float4*>(seg_state + at * D * D + e);
    for (int sg = 0; sg < n_seg; ++sg) {
        const size_t here = at + (size_t)sg * H;
        float4* mine = reinterpret_cast<float4*>(seg_state + here * D * D + e);
        const float4 w = *reinterpret_cast<const float4*>(seg_decay + here * D + i), add = local;
        if (sg + 1 < n_seg) local = *reinterpret_cast<const float4*>(seg_state + (here + H) * D * D + e);
        *mine = cur;
        cur.x = fmaf(w.x, cur.x, add.x);
        cur.y = fmaf(w.y, cur.y, add.y);
        cur.z = fmaf(w.z, cur.z, add.z);
        cur.w = fmaf(w.w, cur.w, add.w);
    }
    *S = cur;
}

LLOGOS_EXPORT int llogos_wkv64(void* y, int out_dtype, const float* r, const float* k, const float* v, const float* d,
                               const float* gate, int ld, int parts, long long part_stride, int d_parts, long long d_part_stride,
                               const float* w0, const float* u, const float* g, float eps, float* state, long long state_stride,
                               long long prev_offset, const float* h_in, int W, const int* slots, const int* cu, int B, int H,
                               int n_seg, int seg_len, float* seg_state, float* seg_decay, hipStream_t stream) {
    if (B <= 0 || H <= 0 || ld < H * kWkvDim || parts < 1 || d_parts < 1 || n_seg < 1) return LLOGOS_BAD_ARGUMENT;
    if (n_seg > 1 && (!cu || seg_len < 1 || !seg_state || !seg_decay)) return LLOGOS_BAD_ARGUMENT;
    if (out_dtype != DT_F32 && out_dtype != DT_BF16) return LLOGOS_BAD_ARGUMENT;
    if ((state_stride & 3) || ((uintptr_t)state & 15) || B > 65535) return LLOGOS_UNSUPPORTED;
    const dim3 grid((H + kWkvWaves - 1) / kWkvWaves, B, n_seg);
#define WKV(MODE, C, TO) wkv64_kernel<MODE, C, TO><<<grid, kWkvWaves * kWave, 0, stream>>>((TO*)y, r, k, v, d, gate, ld, parts, (size_t)part_stride, \
        d_parts, (size_t)d_part_stride, w0, u, g, eps, state, (size_t)state_stride, (size_t)prev_offset, h_in, W, slots, cu, H, n_seg, seg_len, \
        seg_state, seg_decay)
    if (n_seg == 1) {
        if (!cu) { if (out_dtype == DT_F32) WKV(0, 1, float); else WKV(0, 1, bf16_t); }
        else if (out_dtype == DT_F32) WKV(0, 8, float); else WKV(0, 8, bf16_t);
    } else {
        WKV(1, 8, float);
        wkv64_combine_kernel<<<dim3(H, B, kWkvDim * kWkvDim / 1024), 256, 0, stream>>>(state, (size_t)state_stride, slots, seg_state, seg_decay, H, n_seg);
        if (out_dtype == DT_F32) WKV(2, 8, float); else WKV(2, 8, bf16_t);
    }
#undef WKV
    return LLOGOS_LAUNCH_CHECK();
}
