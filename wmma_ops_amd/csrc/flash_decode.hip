// Flash-attention forward for decoding shapes on gfx950: at most 32 query rows per key/value
// head (the query heads of a group times the queries of each), no causal mask, dense layout.
//
// The work is a read of K and V, once.  What bounds it is how many bytes a CU keeps in flight
// and how evenly the reads spread, so a wave here is on its own until the end: it takes every
// W-th step of 32 keys of its workgroup's key range, with the next step's 16 KB (D = 128) in
// flight in registers while a step is computed -- no LDS ring, no barrier in the loop.
//
//  * S^T = K Q^T on v_mfma_f32_16x16x32_f16: a lane loads 16 bytes of key row lane%16, d quarter
//    lane/16 of each 32 of d: the A operand as it arrives.  A lane then owns query lane%16 and
//    keys 4 (lane/16) + 0..3 of each 16-key block.
//  * O^T += V^T P^T: those 8 probabilities are the B operand of one MFMA if its K index runs
//    over keys {4 q .. 4 q + 3, 16 + 4 q .. 16 + 4 q + 3} in quarter q, so V rows are loaded in
//    that order -- 16 bytes (8 columns) of 8 key rows per lane -- and transposed 8x8 in
//    registers (32 v_perm); MFMA j holds columns 8 i + j.  P never leaves its lane.
//  * Softmax as in the forward kernel: base 2, fp32, a stale running max that moves only when
//    a lane's sum shows that some probability could leave fp16's range.
//  * The waves' maxima, sums and O meet in LDS once; with one chunk of keys the output is final,
//    else unnormalised partials go to the workspace for flash_combine_kernel.
#include <algorithm>

#include "common.hpp"
#include "flash_sched.hpp"
#include "kernels.hpp"
#include "plan.hpp"

namespace wmma_amd {

namespace {

constexpr float kNegInfD = -__builtin_huge_valf();
constexpr int FD_KEYS = 32;  // keys per step

struct DecodeArgs {
    const f16* Q;
    const f16* K;
    const f16* V;
    f16* O;
    float* lse;
    int rows;         // query rows per key/value head
    int heads;        // key/value heads per batch entry (a unit is one of them)
    int Sk, dr;
    ChunkStrides q, k, v;  // k.row == v.row; O is contiguous
    FastDiv div_heads;
    float scale_log2;
    int chunk;        // steps per workgroup
    float* o_part;    // [chunks][units * rows][dr], nullptr: one chunk, final output
    float* ml_part;   // [chunks][units * rows][2]
};

constexpr int FD_WAVES = 4;
constexpr int FD_MAX_ROWS = 32;

// Registers decide the waves per SIMD: two steps of K and V (128 a lane at D = 128, 256 at
// D = 256) beside Q, O and the transposed V.  Four waves to a workgroup measured level with
// or ahead of eight (8 x 32 / 8 heads, 4001 keys, the fastest split of each: 26.4 us against
// 27.4; 32 x 40 / 8 heads, 16384 keys: 302 against 308): two workgroups to a CU overlap one's
// start and end with the other's loads.
template <int D, int MB>
struct FdCfg {
    static constexpr int WAVES = FD_WAVES;
    static constexpr int KU = D / 32;               // 16-byte loads per key row and lane
    static constexpr int VH = D > 128 ? 2 : 1;      // 128-column halves of V
    static constexpr int VC = D >= 128 ? 8 : 4;     // columns per lane of a V load
    static constexpr int NO = VH * VC;              // 16-row output blocks of O^T
    // The next step in flight while one is computed; at D = 256 with 32 rows the registers
    // hold one step (without spills 37 us against 46: 2 x 16 / 2 heads, 4 queries, 9000 keys).
    static constexpr bool AHEAD = D <= 128 || MB == 1;
    static constexpr int PER_SIMD = D <= 128 && MB == 1 ? 2 : 1;
};

template <int D>
struct FdK {
    u32x4 x[2][D / 32];
};
template <int D>
struct FdV {
    u32x4 x[D > 128 ? 2 : 1][8];  // D = 64: the low 8 bytes
};

template <int D, int MB>
__global__ void __launch_bounds__((FdCfg<D, MB>::WAVES * kWave))
__attribute__((amdgpu_waves_per_eu(FdCfg<D, MB>::PER_SIMD)))
flash_decode_kernel(DecodeArgs p) {
    using C = FdCfg<D, MB>;
    constexpr int W = C::WAVES, ROWS = 16 * MB, LDR = D + 1;
    __shared__ float red[W][ROWS][LDR];
    __shared__ float red_m[W][ROWS], red_l[W][ROWS];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4, r16 = lane & 15;
    const int unit = blockIdx.x;
    const int Sk = p.Sk, dr = p.dr;
    const int qs = p.q.row_elems(), ks = p.k.row_elems();
    const float c = p.scale_log2;
    const int b = div_by(p.div_heads, unit), hk = unit - b * p.heads;
    const f16* Kb = p.K + p.k.at(b, hk, 0);
    const f16* Vb = p.V + p.v.at(b, hk, 0);

    // Query row 16 mb + lane%16, d = 32 u + 8 q + 0..7 (zeros past the rows and past dr).
    f16x8 qf[MB][C::KU];
    {
        const __amdgpu_buffer_rsrc_t rs = make_rsrc(p.Q + p.q.at(b, hk, 0));
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int u = 0; u < C::KU; ++u) {
                const int row = 16 * mb + r16, d = 32 * u + 8 * q;
                qf[mb][u] = as_f16x8(
                    buf_load16(rs, row < p.rows && d < dr ? (uint32_t)((row * qs + d) * 2) : kOobOffset));
            }
    }

    const int nsteps = (Sk + FD_KEYS - 1) / FD_KEYS;
    const int s0 = (int)blockIdx.y * p.chunk + wave;
    const int s1 = min(nsteps, ((int)blockIdx.y + 1) * p.chunk);
    // Loads of a step past the range go out of bounds (zeros, no memory request), so the loop
    // has no branch around them.
    auto tile = [&](const f16* base, int s) {
        return make_rsrc(base + (int64_t)min(s, nsteps - 1) * FD_KEYS * ks);
    };
    auto load_k = [&](int s, FdK<D>& S) {
        const int left = s < s1 ? Sk - s * FD_KEYS : 0;
        const __amdgpu_buffer_rsrc_t rk = tile(Kb, s);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int u = 0; u < C::KU; ++u) {
                const int key = 16 * kb + r16, d = 32 * u + 8 * q;
                S.x[kb][u] = buf_load16_nt(rk, key < left && d < dr ? (uint32_t)((key * ks + d) * 2)
                                                                   : kOobOffset);
            }
    };
    auto load_v = [&](int s, FdV<D>& S) {
        const int left = s < s1 ? Sk - s * FD_KEYS : 0;
        const __amdgpu_buffer_rsrc_t rv = tile(Vb, s);
#pragma unroll
        for (int vh = 0; vh < C::VH; ++vh)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int key = 16 * (e >> 2) + 4 * q + (e & 3);
                const int d = 128 * vh + C::VC * r16;
                const uint32_t off = key < left && d < dr ? (uint32_t)((key * ks + d) * 2) : kOobOffset;
                if constexpr (C::VC == 8) {
                    S.x[vh][e] = buf_load16_nt(rv, off);
                } else {
                    const u32x2 x = buf_load8(rv, off);
                    S.x[vh][e] = u32x4{x[0], x[1], 0, 0};
                }
            }
    };

    f32x4 O[C::NO][MB];
#pragma unroll
    for (int j = 0; j < C::NO; ++j)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) O[j][mb] = f32x4{};
    float m_run[MB], l_run[MB];  // this lane's query: running max; sum over this lane's keys
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        m_run[mb] = kNegInfD;
        l_run[mb] = 0.0f;
    }

    auto compute = [&](int s, const FdK<D>& SK, const FdV<D>& SV) {
        if (s >= s1) return;  // uniform
        f32x4 sc[MB][2];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                sc[mb][kb] = f32x4{};
#pragma unroll
                for (int u = 0; u < C::KU; ++u)
                    sc[mb][kb] = mfma16(as_f16x8(SK.x[kb][u]), qf[mb][u], sc[mb][kb]);
            }
        if ((s + 1) * FD_KEYS > Sk) {
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (s * FD_KEYS + 16 * (e >> 2) + 4 * q + (e & 3) >= Sk)
                        sc[mb][e >> 2][e & 3] = kNegInfD;
        }
        f16x8 P[MB];
        float sum[MB];
        auto exps = [&](int mb, float m) {
            float t[2] = {0.0f, 0.0f};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float pv = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[mb][e >> 2][e & 3], c, -m));
                t[e & 1] += pv;
                P[mb][e] = (f16)pv;
            }
            sum[mb] = t[0] + t[1];
        };
        bool need = false;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const bool fresh = m_run[mb] == kNegInfD;
            exps(mb, fresh ? 0.0f : m_run[mb]);
            need |= fresh || !(sum[mb] <= 32768.0f);  // also inf and NaN
        }
        if (__builtin_amdgcn_ballot_w64(need) != 0) {  // wave-uniform, rare
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                float mx = kNegInfD;
#pragma unroll
                for (int e = 0; e < 8; ++e) mx = fmaxf(mx, sc[mb][e >> 2][e & 3]);
                mx = fmaxf(mx, __shfl_xor(mx, 16));
                mx = fmaxf(mx, __shfl_xor(mx, 32));
                const float mn = fmaxf(m_run[mb], mx * c);
                const float alpha =
                    m_run[mb] == kNegInfD ? 0.0f : __builtin_amdgcn_exp2f(m_run[mb] - mn);
                m_run[mb] = mn;
                l_run[mb] *= alpha;
                exps(mb, mn == kNegInfD ? 0.0f : mn);
#pragma unroll
                for (int j = 0; j < C::NO; ++j) O[j][mb] *= alpha;
            }
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) l_run[mb] += sum[mb];
#pragma unroll
        for (int vh = 0; vh < C::VH; ++vh) {
            u32x4 vt[8];
            if constexpr (C::VC == 8) {
                transpose8x8(SV.x[vh], vt);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int d = 0; d < 4; ++d)
                        vt[j][d] = __builtin_amdgcn_perm(SV.x[vh][2 * d + 1][j >> 1], SV.x[vh][2 * d][j >> 1],
                                                         (j & 1) ? kPermHi : kPermLo);
            }
#pragma unroll
            for (int j = 0; j < C::VC; ++j)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
                    O[C::VC * vh + j][mb] = mfma16(as_f16x8(vt[j]), P[mb], O[C::VC * vh + j][mb]);
        }
    };

    FdK<D> K0;
    load_k(s0, K0);
    FdV<D> V0;
    if constexpr (C::AHEAD) {
        FdK<D> K1;
        FdV<D> V1;
        load_v(s0, V0);
        for (int s = s0; s < s1; s += 2 * W) {
            load_k(s + W, K1);
            load_v(s + W, V1);
            compute(s, K0, V0);
            load_k(s + 2 * W, K0);
            load_v(s + 2 * W, V0);
            compute(s + W, K1, V1);
        }
    } else {
        for (int s = s0; s < s1; s += W) {
            load_v(s, V0);
            compute(s, K0, V0);
            load_k(s + W, K0);
        }
    }

    // The waves meet: O^T block j holds query lane%16, d = 128 (j / VC) + VC (4 q + r) + j % VC.
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        float l = l_run[mb];
        l += __shfl_xor(l, 16);
        l += __shfl_xor(l, 32);
        if (q == 0) {
            red_m[wave][16 * mb + r16] = m_run[mb];
            red_l[wave][16 * mb + r16] = l;
        }
#pragma unroll
        for (int j = 0; j < C::NO; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                red[wave][16 * mb + r16][128 * (j / C::VC) + C::VC * (4 * q + r) + j % C::VC] = O[j][mb][r];
    }
    __syncthreads();
    const int dq = dr / 4;
    for (int e = tid; e < p.rows * dq; e += W * kWave) {
        const int row = e / dq, d = 4 * (e - row * dq);
        float m = red_m[0][row];
#pragma unroll
        for (int w = 1; w < W; ++w) m = fmaxf(m, red_m[w][row]);
        float l = 0.0f, acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const float mw = red_m[w][row];
            const float a = mw == kNegInfD ? 0.0f : __builtin_amdgcn_exp2f(mw - m);
            l += a * red_l[w][row];
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] += a * red[w][row][d + i];
        }
        const int64_t r = (int64_t)unit * p.rows + row;
        if (p.o_part) {
            const int64_t z = (int64_t)blockIdx.y * gridDim.x * p.rows + r;
            if (d == 0) {
                p.ml_part[2 * z] = m;
                p.ml_part[2 * z + 1] = l;
            }
            *reinterpret_cast<float4*>(p.o_part + z * dr + d) = make_float4(acc[0], acc[1], acc[2], acc[3]);
        } else {
            const float inv = l > 0.0f ? 1.0f / l : 0.0f;
            f16x4 o;
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = (f16)(acc[i] * inv);
            *reinterpret_cast<f16x4*>(p.O + r * dr + d) = o;
            if (p.lse && d == 0)
                p.lse[r] = l > 0.0f ? (m + __builtin_amdgcn_logf(l)) * 0.6931471805599453f
                                    : __builtin_huge_valf();
        }
    }
}

template <int D>
void launch_decode_d(const DecodeArgs& a, dim3 grid, hipStream_t stream) {
    const dim3 block(FD_WAVES * kWave);
    if (a.rows <= 16)
        hipLaunchKernelGGL((flash_decode_kernel<D, 1>), grid, block, 0, stream, a);
    else
        hipLaunchKernelGGL((flash_decode_kernel<D, 2>), grid, block, 0, stream, a);
}

}  // namespace

// Two row blocks against a step or less per wave leave this kernel its prologue and the merge of
// its waves: 32 rows, D = 128, 4 x 32 heads, 4 / 64 / 128 / 200 keys 6.8 / 7.0 / 7.9 / 8.8 us here,
// 5.6 / 5.4 / 6.5 / 9.0 on the general kernel; D = 64 level.
bool flash_decode_takes(int Sq, int Sk, int D, bool causal) {
    if (causal || Sq < 1 || Sq > FD_MAX_ROWS) return false;
    return Sq <= 16 || D <= 64 || Sk > FD_WAVES * FD_KEYS;
}

// Chunks of the key range: 256 keys or more each, down to 96 while fewer than 64 workgroups
// run.  The time of a split, read off a sweep of 1-64 chunks at 17 shapes (2-512 units,
// 318-32768 keys, D = 64-256): the reads at 24.5 KB/us per busy CU and at most 6.2 TB/s; past
// one wave of workgroups the busiest CU sets the pace (80 units, 5408 keys: 3 chunks 32 us, 4
// chunks -- 320 workgroups -- 42 us); two chunks or more add the merge and their partial
// sums.  The split that fills the CUs once stays unless another is 1% better.
int flash_decode_split(int64_t units, int Sq, int Sk, int D, int num_cus) {
    const int steps = ceil_div(Sk, FD_KEYS);
    const double mb = (double)units * Sk * D * 4e-6;
    const int few = (int)std::min<int64_t>(std::max<int64_t>(64 / units, 1), Sk / 96);
    const int most = std::min(64, std::max({Sk / 256, few, 1}));
    const int fill = (int)std::min<int64_t>(std::max<int64_t>(num_cus / units, 1), most);
    auto time = [&](int z) {
        const int64_t wgs = units * z;
        const double rate = std::min(6.2, 0.0245 * (double)std::min<int64_t>(wgs, num_cus));
        const double uneven =
            wgs > num_cus ? (double)(ceil_div64(wgs, num_cus) * num_cus) / (double)wgs : 1.0;
        const double t = 2.5 + uneven * mb / rate;
        return z > 1 ? t + 5.0 + 0.15 * z + (double)z * units * Sq * D * 8e-6 / 5.0 : t;
    };
    auto chunks = [&](int z) { return ceil_div(steps, ceil_div(steps, z)); };
    int best = chunks(fill);
    double best_t = time(best);
    for (int z = 1; z <= most; z = z < 8 ? z + 1 : z + z / 8) {
        const double t = time(chunks(z));
        if (t < best_t * 0.99) {
            best_t = t;
            best = chunks(z);
        }
    }
    return best;
}

// Steps of a chunk; the chunks of a split hold ceil(steps / chunk).
static int decode_chunk(int Sk, int split) { return ceil_div(ceil_div(Sk, FD_KEYS), split); }

size_t flash_decode_workspace_bytes(int64_t units, int Sq, int Sk, int D, int split) {
    if (split <= 1) return 0;
    const int z = ceil_div(ceil_div(Sk, FD_KEYS), decode_chunk(Sk, split));
    return (size_t)z * units * Sq * (size_t)(D + 2) * sizeof(float);
}

hipError_t launch_flash_decode(const FlashLaunch& f, hipStream_t stream) {
    DecodeArgs a{};
    a.Q = static_cast<const f16*>(f.Q);
    a.K = static_cast<const f16*>(f.K);
    a.V = static_cast<const f16*>(f.V);
    a.O = static_cast<f16*>(f.O);
    a.lse = f.lse;
    a.rows = f.Sq;
    a.heads = f.H;
    a.q = chunks_of(f.q);
    a.k = chunks_of(f.k);
    a.v = chunks_of(f.v);
    a.div_heads = fast_div(f.H);
    a.Sk = f.Sk;
    a.dr = f.D;
    a.scale_log2 = f.scale * 1.4426950408889634f;
    const int64_t units = (int64_t)f.B * f.H;
    a.chunk = decode_chunk(f.Sk, f.kv_split);
    const int z = ceil_div(ceil_div(f.Sk, FD_KEYS), a.chunk);
    const int64_t rows = units * f.Sq;
    if (z > 1) {
        a.o_part = static_cast<float*>(f.workspace);
        a.ml_part = a.o_part + (int64_t)z * rows * f.D;
    }
    const dim3 grid((unsigned)units, z);
    if (f.D > 128)
        launch_decode_d<256>(a, grid, stream);
    else if (f.D > 64)
        launch_decode_d<128>(a, grid, stream);
    else
        launch_decode_d<64>(a, grid, stream);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || z == 1) return e;
    return launch_flash_combine(a.o_part, a.ml_part, z, rows, f.D, f.O, f.lse, stream);
}

}  // namespace wmma_amd
