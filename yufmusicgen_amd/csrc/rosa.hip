// ROSA Householder memory scan for gfx950 (MI355X).
//
// Semantics: yufmusicgen/model.py:260-288 (reference recurrence) and the read
// of model.py:303-311 / yufmusicgen/cuda/rosa_householder.cu:30-101:
//     m_t    = lambda * H(m_{t-1}) + e_t,   e_t = sigmoid(write_t) tanh(cand_t)
//     read_t = H(m_t) [* sigmoid(read_raw_t)],     H(x) = x - 2 (x.u) u.
//
// The transition diag(lambda) H = diag(lambda) - 2 (lambda u) u^T is diagonal
// plus rank one, so with p_t = u.m_{t-1} the recurrence is
//     m_t = lambda (m_{t-1} - 2 p_t u) + e_t.
// Over a chunk of C tokens starting from m_0 (1-based tau):
//     m_tau = y_tau - 2 c_tau,  y_tau = lambda^tau m_0 + z_tau,
//     z_tau = lambda z_{tau-1} + e_tau (z_0 = 0),  c_tau = lambda (c_{tau-1} + p_tau u),
// and the projections solve a lower-triangular Toeplitz system
//     p_tau + 2 sum_{s<tau} kappa_{tau-s} p_s = f_tau := u.y_{tau-1},
//     kappa_n = sum_j u_j^2 lambda_j^n,   p = L f,  L[tau][s] = ell_{tau-s},
//     ell_0 = 1, ell_n = -2 sum_{k=1..n} kappa_k ell_{n-k}.
// So the only cross-channel reductions are the C+1 dot products f (one batch
// per chunk), not one wave reduction per token as in the direct recurrence.
//
// One workgroup per stream, 1 consumer wave + 6 producer waves, three LDS
// stages in flight (chunk i+1 staged, chunk i solved, chunk i-1 emitted):
//   producers, A(i+1): turn chunk i+1's pre-activations (loaded one iteration
//       earlier with bounds-checked buffer loads) into e and the gate in LDS --
//       or take e and the gate as computed by the model's input projection --
//       and run the per-channel z recurrence;
//   consumer, B(i):   f = u.(lambda^tau m_0 + z_tau) for tau = 0..C (per-lane
//       partials, transposed through LDS), p = L f, then the chunk-end state;
//   producers, O(i-1): per channel, m_tau = lambda (m_{tau-1} - 2 p_tau u) + e_tau
//       with the now-known p, and read_tau = (m_tau - 2 p_{tau+1} u) g_tau.
// All waves meet at one barrier per chunk.
//
// D in {64, 128, 256} takes the segment kernel further down instead: 32-token
// chunks with the same algebra, every phase spread over the workgroup, and long
// sequences cut into segments.
#include "common.h"
#include "kernels.h"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <tuple>
#include <utility>

namespace yuf {
namespace {

constexpr int kWave = 64;
// Waves w and w + 4 of a workgroup share a SIMD: the consumer (wave 0) keeps its
// SIMD to itself (wave 4 only joins the barriers), six producers take waves
// 1-3 and 5-7.
constexpr int kProducerWaves = 6;
constexpr int kThreads = 8 * kWave;
constexpr int kStages = 3;

template <int EPL>
struct Cfg {
    static constexpr int C = EPL <= 2 ? 16 : (EPL == 4 ? 8 : (EPL == 8 ? 4 : 2));  // tokens per chunk
    static constexpr int DP = EPL * kWave;                                          // padded channels
    static constexpr int ZS = C + 1;          // odd row stride of the transposed z / partial arrays
    static constexpr int CH = (DP + kProducerWaves - 1) / kProducerWaves;  // channels per producer wave
    static constexpr int CPL = (CH + kWave - 1) / kWave;                   // channels per producer lane
    static constexpr int kItems = (C * CH + kWave - 1) / kWave;            // (token, channel) loads per lane
};

// LDS-only ordering between lanes of one wave (no s_barrier).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int EPL>
__global__ void __launch_bounds__(kThreads) rosa_scan_kernel(RosaParams p) {
    using K = Cfg<EPL>;
    constexpr int C = K::C, DP = K::DP, ZS = K::ZS, CH = K::CH, CPL = K::CPL;
    __shared__ __attribute__((aligned(16))) float ew[kStages][C * DP];  // e_tau   [tau][c]
    __shared__ __attribute__((aligned(16))) float gt[kStages][C * DP];  // gate    [tau][c]
    __shared__ float zt[kStages][DP * ZS];                              // z_tau   [c][tau], tau = 0..C
    __shared__ float pv[kStages][ZS];                                   // p_{tau+1}, tau = 0..C
    __shared__ float m0b[kStages][DP];                                  // chunk-start state
    __shared__ float lam_s[DP], u_s[DP];
    // Consumer-only: per-lane partial dot products [lane][tau], f, and the Toeplitz
    // inverse ell, in double: ell alternates in sign with |ell_n| up to 2 when the
    // decay is near 1, so p = L f adds up to C rounding errors of f with weight 2.
    __shared__ double part[kWave * ZS];
    __shared__ double fv[ZS], ell[ZS];

    const int bb = blockIdx.x;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int D = p.D;
    const int slot = p.slot ? p.slot[bb] : bb;
    const bool gated = p.read_raw != nullptr || p.e_pre != nullptr;
    const int n_chunks = (p.T + C - 1) / C;

    // ------------------------------------------------------------ producers
    const int pw = wave < 4 ? wave - 1 : wave - 2;  // producer index on waves 1-3, 5-7
    const bool producer = wave != 0 && wave != 4;
    const bool prepared = p.e_pre != nullptr;
    // Next chunk's inputs, loaded one iteration ahead: (cand, write, read_raw) or,
    // prepared, (e, gate).  Every load is issued; an input that is not needed
    // has a zero-size descriptor and reads 0 without touching memory.
    float in0[K::kItems], in1[K::kItems], in2[K::kItems];
    auto load_in = [&](int ch) {
        const int t0 = ch * C, nt = min(C, p.T - t0);
        const size_t base = (size_t)(bb * p.T + t0) * p.ld;
        const uint32_t bytes = (uint32_t)(((nt - 1) * p.ld + D) * 4);
        const auto r0 = make_rsrc((prepared ? p.e_pre : p.cand) + base, bytes);
        const auto r1 = make_rsrc((prepared ? p.g_pre : p.write) + base, bytes);
        const auto r2 = make_rsrc(gated && !prepared ? p.read_raw + base : p.cand + base,
                                  gated && !prepared ? bytes : 0u);
#pragma unroll
        for (int it = 0; it < K::kItems; ++it) {
            const int q = lane + it * kWave;
            const int tau = q / CH, c = pw * CH + (q - tau * CH);
            const uint32_t off = (q < C * CH && c < D && tau < nt) ? (uint32_t)(tau * p.ld + c) * 4u : kBufferOob;
            in0[it] = buf_load(r0, off);
            in1[it] = buf_load(r1, off);
            in2[it] = buf_load(r2, off);
        }
    };
    auto stage_in = [&](int ch) {  // A(ch), from the registers load_in(ch) filled
        const int s = ch % kStages;
#pragma unroll
        for (int it = 0; it < K::kItems; ++it) {
            const int q = lane + it * kWave;
            const int tau = q / CH, c = pw * CH + (q - tau * CH);
            if (q < C * CH && c < DP) {
                float e, gv;
                if (prepared) {
                    e = in0[it];
                    gv = in1[it];
                } else {
                    // tanh(x) = 1 - 2 / (e^{2x} + 1); sigmoid(x) = 1 / (1 + e^{-x}).  Out-of-range
                    // tokens and channels read 0 and give e = 0.
                    const float th = 1.0f - 2.0f * __frcp_rn(__expf(2.0f * in0[it]) + 1.0f);
                    e = th * __frcp_rn(1.0f + __expf(-in1[it]));
                    gv = gated ? __frcp_rn(1.0f + __expf(-in2[it])) : 1.0f;
                }
                ew[s][tau * DP + c] = e;
                gt[s][tau * DP + c] = gv;
            }
        }
        wave_lds_sync();
#pragma unroll
        for (int k = 0; k < CPL; ++k) {
            const int cc = lane + k * kWave;
            const int c = pw * CH + cc;
            if (cc < CH && c < DP) {
                const float lam = lam_s[c];
                float z = 0.0f;
                zt[s][c * ZS] = 0.0f;
#pragma unroll
                for (int tau = 0; tau < C; ++tau) {
                    z = fmaf(lam, z, ew[s][tau * DP + c]);
                    zt[s][c * ZS + tau + 1] = z;
                }
            }
        }
    };
    auto emit = [&](int ch) {  // O(ch)
        const int s = ch % kStages, t0 = ch * C, nt = min(C, p.T - t0);
        const size_t obase = (size_t)(bb * p.T + t0) * D;
        const auto ro = make_rsrc(p.read_out + obase, (uint32_t)(nt * D * 4));
#pragma unroll
        for (int k = 0; k < CPL; ++k) {
            const int cc = lane + k * kWave;
            const int c = pw * CH + cc;
            if (cc < CH && c < DP) {
                const float lam = lam_s[c], u = u_s[c];
                float m = m0b[s][c];
                // All C steps run (tokens past nt have e = 0 and are not stored), so
                // the LDS reads are independent of the chain and issue up front.
#pragma unroll
                for (int tau = 0; tau < C; ++tau) {
                    m = fmaf(lam, fmaf(-2.0f * pv[s][tau], u, m), ew[s][tau * DP + c]);
                    const float rv = fmaf(-2.0f * pv[s][tau + 1], u, m) * gt[s][tau * DP + c];
                    buf_store(rv, ro, (c < D && tau < nt) ? (uint32_t)(tau * D + c) * 4u : kBufferOob);
                }
            }
        }
    };

    // ------------------------------------------------------------- consumer
    float lam[EPL], u[EPL], m0[EPL];
    if (wave == 0) {
        float nrm = 0.0f;
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
            const int c = lane + e * kWave;
            const bool ok = c < D;
            u[e] = ok ? p.direction[c] : 0.0f;
            lam[e] = ok ? p.decay[c] : 0.0f;
            m0[e] = (ok && p.memory_in) ? p.memory_in[(size_t)slot * D + c] : 0.0f;
            nrm = fmaf(u[e], u[e], nrm);
        }
        if (p.raw_params) {
            // Model path: u = householder / max(|householder|, 1e-12), lambda = sigmoid(decay)
            // (model.py:300-301).
            const float inv = 1.0f / fmaxf(sqrtf(wave_sum(nrm)), 1e-12f);
#pragma unroll
            for (int e = 0; e < EPL; ++e) {
                const int c = lane + e * kWave;
                u[e] *= inv;
                lam[e] = c < D ? 1.0f / (1.0f + expf(-lam[e])) : 0.0f;
            }
        }
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
            lam_s[lane + e * kWave] = lam[e];
            u_s[lane + e * kWave] = u[e];
        }
        // kappa_n = sum_j u_j^2 lambda_j^n, n = 1..C, then the Toeplitz inverse ell.
        {
            double pw_[EPL];
#pragma unroll
            for (int e = 0; e < EPL; ++e) pw_[e] = (double)u[e] * u[e];
            for (int n = 1; n <= C; ++n) {
                double acc = 0.0;
#pragma unroll
                for (int e = 0; e < EPL; ++e) {
                    pw_[e] *= lam[e];
                    acc += pw_[e];
                }
                part[lane * ZS + n] = acc;
            }
            wave_lds_sync();
            if (lane >= 1 && lane <= C) {
                double acc = 0.0;
                for (int k = 0; k < kWave; ++k) acc += part[k * ZS + lane];
                fv[lane] = acc;  // kappa_lane
            }
            wave_lds_sync();
            if (lane == 0) {
                ell[0] = 1.0;
                for (int n = 1; n <= C; ++n) {
                    double acc = 0.0;
                    for (int k = 1; k <= n; ++k) acc = fma(fv[k], ell[n - k], acc);
                    ell[n] = -2.0 * acc;
                }
            }
            wave_lds_sync();
        }
        wait_vmem();
    }
    lds_barrier();  // lam_s / u_s visible to the producers
    if (producer && n_chunks > 0) {
        load_in(0);
        stage_in(0);
        if (n_chunks > 1) load_in(1);
    }
    lds_barrier();

    for (int i = 0; i <= n_chunks; ++i) {
        if (wave == 0) {
            if (i < n_chunks) {
                const int s = i % kStages, nt = min(C, p.T - i * C);
                // f_{tau+1} = u . (lambda^tau m_0 + z_tau), tau = 0..C: per-lane partials.
                float y[EPL];
#pragma unroll
                for (int e = 0; e < EPL; ++e) y[e] = m0[e];
                for (int tau = 0; tau <= C; ++tau) {
                    double acc = 0.0;
#pragma unroll
                    for (int e = 0; e < EPL; ++e) {
                        const double ud = u[e];
                        acc = fma(ud, (double)y[e], fma(ud, (double)zt[s][(lane + e * kWave) * ZS + tau], acc));
                        y[e] *= lam[e];
                    }
                    part[lane * ZS + tau] = acc;
                }
                wave_lds_sync();
                // Sums over the 64 lanes' partials and the Toeplitz products use
                // independent accumulators: these chains are the scan's critical path.
                if (lane <= C) {
                    double a8[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
                    for (int k = 0; k < kWave; k += 8)
#pragma unroll
                        for (int m = 0; m < 8; ++m) a8[m] += part[(k + m) * ZS + lane];
                    fv[lane] = ((a8[0] + a8[1]) + (a8[2] + a8[3])) + ((a8[4] + a8[5]) + (a8[6] + a8[7]));
                }
                wave_lds_sync();
                if (lane <= C) {
                    double a4[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                    for (int sg = 0; sg <= C; ++sg) {
                        const double coef = sg <= lane ? ell[sg <= lane ? lane - sg : 0] : 0.0;
                        a4[sg & 3] = fma(coef, fv[sg], a4[sg & 3]);
                    }
                    pv[s][lane] = (float)((a4[0] + a4[1]) + (a4[2] + a4[3]));
                }
#pragma unroll
                for (int e = 0; e < EPL; ++e) m0b[s][lane + e * kWave] = m0[e];
                wave_lds_sync();
                // State after the chunk's nt real tokens:
                // m_nt = lambda^nt m_0 + z_nt - 2 sum_{s<=nt} p_s lambda^{nt-s+1} u.
                float acc[EPL], pwr[EPL];
#pragma unroll
                for (int e = 0; e < EPL; ++e) { acc[e] = 0.0f; pwr[e] = m0[e]; }
#pragma unroll
                for (int sg = 0; sg < C; ++sg) {
                    const float ps = pv[s][sg];
#pragma unroll
                    for (int e = 0; e < EPL; ++e) {
                        if (sg < nt) {
                            acc[e] = lam[e] * fmaf(ps, u[e], acc[e]);
                            pwr[e] *= lam[e];
                        }
                    }
                }
#pragma unroll
                for (int e = 0; e < EPL; ++e)
                    m0[e] = fmaf(-2.0f, acc[e], pwr[e] + zt[s][(lane + e * kWave) * ZS + nt]);
            }
        } else if (producer) {
            if (i >= 1) emit(i - 1);
            if (i + 1 < n_chunks) {
                stage_in(i + 1);
                if (i + 2 < n_chunks) load_in(i + 2);
            }
        }
        lds_barrier();
    }
    if (wave == 0 && p.memory_out) {
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
            const int c = lane + e * kWave;
            if (c < D) p.memory_out[(size_t)slot * D + c] = m0[e];
        }
    }
}

}  // namespace


// Single-token step (T = 1, decode): one wave per stream, EPL channels per
// lane, the direct recurrence with its two projections (u.m_{t-1} and u.m_t)
// summed in double across the wave, and the gates computed from the raw
// pre-activations in place (the same float expressions as the scan's
// activation path) -- one kernel, no separate gate pass.
template <int EPL>
__global__ void __launch_bounds__(256) rosa_step_kernel(RosaParams p) {
    const int bb = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (bb >= p.B) return;
    const int D = p.D;
    const int slot = p.slot ? p.slot[bb] : bb;
    const bool prepared = p.e_pre != nullptr;
    const bool gated = p.read_raw != nullptr || prepared;
    const size_t base = (size_t)bb * p.ld;
    float u[EPL], lam[EPL], m[EPL], ev[EPL], gv[EPL];
    float nrm = 0.0f;
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
        const int c = lane + e * kWave;
        const bool ok = c < D;
        u[e] = ok ? p.direction[c] : 0.0f;
        lam[e] = ok ? p.decay[c] : 0.0f;
        m[e] = (ok && p.memory_in) ? p.memory_in[(size_t)slot * D + c] : 0.0f;
        ev[e] = ok ? (prepared ? p.e_pre : p.cand)[base + c] : 0.0f;
        gv[e] = ok ? (prepared ? p.g_pre : p.write)[base + c] : 0.0f;
        nrm = fmaf(u[e], u[e], nrm);
    }
    float rr[EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
        const int c = lane + e * kWave;
        rr[e] = (c < D && gated && !prepared) ? p.read_raw[base + c] : 0.0f;
    }
    if (p.raw_params) {
        const float inv = 1.0f / fmaxf(sqrtf(wave_sum(nrm)), 1e-12f);
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
            const int c = lane + e * kWave;
            u[e] *= inv;
            lam[e] = c < D ? 1.0f / (1.0f + expf(-lam[e])) : 0.0f;
        }
    }
    if (!prepared) {
#pragma unroll
        for (int e = 0; e < EPL; ++e) {
            const float th = 1.0f - 2.0f * __frcp_rn(__expf(2.0f * ev[e]) + 1.0f);
            ev[e] = th * __frcp_rn(1.0f + __expf(-gv[e]));
            gv[e] = gated ? __frcp_rn(1.0f + __expf(-rr[e])) : 1.0f;
        }
    }
    double f = 0.0;
#pragma unroll
    for (int e = 0; e < EPL; ++e) f = fma((double)u[e], (double)m[e], f);
    const float p1 = (float)wave_sum_f64(f);
    double f2 = 0.0;
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
        m[e] = fmaf(lam[e], fmaf(-2.0f * p1, u[e], m[e]), ev[e]);
        f2 = fma((double)u[e], (double)m[e], f2);
    }
    const float p2 = (float)wave_sum_f64(f2);
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
        const int c = lane + e * kWave;
        if (c < D) {
            p.read_out[(size_t)bb * D + c] = fmaf(-2.0f * p2, u[e], m[e]) * gv[e];
            if (p.memory_out) p.memory_out[(size_t)slot * D + c] = m[e];
        }
    }
}

// Segmented scan of many segments, carry pass.  With a constant transition A =
// diag(lambda) H, the state after segment s of length L is m_{s+1} = A^L m_s +
// z_s, where z_s is the segment's end state from a zero start (z_0: from the
// true start; row P - 1 of a chain's z rows holds that start).  One workgroup
// per chain walks its P segments and records each segment's start state
// (carry).  D in {64, 128, 256}: blockDim = D * D / 64; thread (h, r) = (tid / D,
// tid % D) keeps the 64 entries of row r in column block h in registers, so the
// 64 lanes of a wave read the same 64 state values (LDS broadcasts).  The P
// steps are the chain, so a step only touches registers and LDS: the z rows are
// staged into LDS in blocks before the steps that use them (no global-load wait
// inside the chain, which would also wait for the carry stores in flight), the
// 64 state values are read before the FMAs (four independent chains), and the
// column blocks' partial sums meet in LDS in a fixed order (~0.5 us a step at D
// = 128).
template <int D>
__global__ void __launch_bounds__(D * D / 64) rosa_carry_kernel(int P, const float *AL, const float *z,
                                                                float *carry) {
    constexpr int kZFloats = 16384;  // staged z rows (64 KB)
    constexpr int nthr = D * D / 64, nb = D / 64;
    __shared__ __attribute__((aligned(16))) float st[2][D];
    __shared__ float part[nb][D];
    __shared__ __attribute__((aligned(16))) float zs[kZFloats];
    const int b = blockIdx.x, tid = threadIdx.x;
    const int h = tid / D, r = tid - h * D;
    float arow[64];
    const float4 *arow4 = reinterpret_cast<const float4 *>(AL + (size_t)r * D + h * 64);
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const float4 a4 = arow4[j];
        arow[4 * j] = a4.x; arow[4 * j + 1] = a4.y; arow[4 * j + 2] = a4.z; arow[4 * j + 3] = a4.w;
    }
    if (tid < D) {
        carry[(size_t)b * P * D + tid] = z[((size_t)b * P + P - 1) * D + tid];
        st[1][tid] = z[(size_t)b * P * D + tid];
    }
    constexpr int zb = kZFloats / D;  // steps per staged block
    for (int s0 = 1; s0 < P; s0 += zb) {
        const int n = min(zb, P - s0);
        const float4 *z4 = reinterpret_cast<const float4 *>(z + ((size_t)b * P + s0) * D);
        float4 *zs4 = reinterpret_cast<float4 *>(zs);
        const int total4 = n * D / 4;
        for (int i0 = 0; i0 < total4; i0 += 8 * nthr) {  // eight loads in flight per thread
            float4 t4[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) t4[u] = z4[min(i0 + u * nthr + tid, total4 - 1)];  // in bounds; extras unused
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int i = i0 + u * nthr + tid;
                if (i < total4) zs4[i] = t4[u];
            }
        }
        // LDS-only barriers: the carry stores below stay in flight across them.
        lds_barrier();
        for (int k = 0; k < n; ++k) {
            const int s = s0 + k, cur = s & 1;
            const size_t v = (size_t)b * P + s;
            if (tid < D) carry[v * D + tid] = st[cur][tid];
            float x[64];
            const float4 *x4 = reinterpret_cast<const float4 *>(st[cur] + h * 64);
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const float4 t = x4[j];
                x[4 * j] = t.x; x[4 * j + 1] = t.y; x[4 * j + 2] = t.z; x[4 * j + 3] = t.w;
            }
            float d4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int j = 0; j < 64; j += 4)
#pragma unroll
                for (int q = 0; q < 4; ++q) d4[q] = fmaf(arow[j + q], x[j + q], d4[q]);
            const float dot = (d4[0] + d4[1]) + (d4[2] + d4[3]);
            if constexpr (nb == 1) {
                st[cur ^ 1][r] = dot + zs[k * D + r];
            } else {
                part[h][r] = dot;
                lds_barrier();
                if (h == 0) {
                    float sum = part[0][r];
#pragma unroll
                    for (int q = 1; q < nb; ++q) sum += part[q][r];
                    st[cur ^ 1][r] = sum + zs[k * D + r];
                }
            }
            lds_barrier();
        }
    }
}

// ---------------------------------------------------------------------------
// Segment form, D in {64, 128, 256}.  A scan is bound by its chain, so the
// chain of a 32-token chunk is cut to what depends on the state: with y_tau =
// lambda^tau m_0 + z_tau run as one recurrence per channel, f_{tau+1} = u.y_tau
// are 32 dot products over the channels (summed in double by all waves at
// once), p = L f one small triangular product, and the states and reads follow
// per channel.  f_1 of a chunk is p_33 of the one before.  Five barriers and
// 2.2, 2.8 and 4.2 us per 32 tokens of one segment at D = 64, 128 and 256, against
// 3.5, 6.3 and 9.1 in rosa_scan_kernel.
//
// Long sequences are cut into segments of L tokens: one launch runs every
// segment but the last to its end state (the first from the true start, the
// others from zero), a second one forms each segment's start state from the
// end states before it, m_{s+1} = A^L m_s + z_s, and runs it again with the
// reads.  Every segment's workgroup walks its own copy of that carry (at most
// kRosaChain steps of ~0.4 us, beside its own loads), which saves the carry's
// launch; above that rosa_carry_kernel runs between the two.
// ---------------------------------------------------------------------------
constexpr int kSegC = 32;       // tokens per chunk
constexpr int kSegEll = 40;     // doubles per chain for ell_0 .. ell_32
constexpr int kRosaChain = 32;  // segments whose carry is walked inside the second launch

struct RosaSegParams {
    int B = 0, T = 0, ld = 0, L = 0, P = 0;
    const float *cand = nullptr, *write = nullptr, *read_raw = nullptr;
    const float *lam = nullptr, *u = nullptr;
    const float *memory_in = nullptr;
    float *memory_out = nullptr;
    const int *slot = nullptr;
    float *read_out = nullptr;
    // [B][P][D]: end states of segments 0 .. P - 2; row P - 1 holds the chain's
    // start state (memory_out may alias memory_in, which the second launch must
    // not read once a chain's last segment may have ended).
    float *z = nullptr;
    const float *AL = nullptr;
    const float *starts = nullptr;  // [B][P][D] start states, or nullptr: walked from z
    double *ell = nullptr;          // [B][kSegEll], P > 1: ell_0 .. ell_32 from the first launch
    float *AL_out = nullptr;        // first launch: A^L to compute in its extra workgroups
};

template <int D>
struct SegCfg {
    static constexpr int NT = D == 64 ? 256 : 512;  // threads: D for the chains, the rest turn inputs into e and gates
    static constexpr int CT = NT - D;
    static constexpr int GL = NT / kSegC;            // lanes per dot product
    static constexpr int H = NT / D;                 // column blocks of the carry product
    static constexpr int W = D / H;                  // its columns per thread
    static constexpr int PS = D + 16;                // doubles per row of partial products
    static constexpr int IT = (kSegC * D / 4 + CT - 1) / CT;  // float4 loads per input thread, chunk and input
    static constexpr int kPowEntries = 4;            // entries of A^L per thread
    static constexpr int kPowWgs = D * D / (kPowEntries * NT);
    static constexpr int kLds = kSegC * PS * 8 + 2 * kSegC * D * 4;  // partial products, e, gates
};

// 1 / x to within a rounding or two, x >= 2^-30 or NaN: inf gives 0.
__device__ __forceinline__ float recip(float x) {
    const float r = __builtin_amdgcn_rcpf(x);
    return x > 0x1p126f ? r : fmaf(fmaf(-x, r, 1.0f), r, r);
}
__device__ __forceinline__ float seg_gate(float x) { return recip(1.0f + __expf(-x)); }
// tanh(x) sigmoid(w) = (E - 1) / ((E + 1) (1 + F)), E = e^{2x}, F = e^{-w}: one
// reciprocal.  tanh is 1 in fp32 from x = 10 on (the comparison keeps NaN); 0 for x = 0.
// Both E + 1 and E - 1 carry a factor 2^-30, which changes no bit of the quotient
// and keeps the product finite for every finite F (without it the result vanished
// below w = -69).
__device__ __forceinline__ float seg_cand(float x, float w) {
    float s;  // 2^-30 in a scalar register (a vector one is a spill at D = 256)
    asm("s_mov_b32 %0, 0x30800000" : "=s"(s));
    const float E = __expf(2.0f * (x > 10.0f ? 10.0f : x));
    return fmaf(E, s, -s) * recip(fmaf(E, s, s) * (1.0f + __expf(-w)));
}

// Sum over aligned groups of G lanes (8 or 16), every lane gets it.
template <int G>
__device__ __forceinline__ double group_sum_f64(double x) {
    static_assert(G == 8 || G == 16, "group size");
    x += dpp_move_f64<dpp::kQuadXor1>(x);
    x += dpp_move_f64<dpp::kQuadXor2>(x);
    x += dpp_move_f64<dpp::kRowHalfMirror>(x);
    if constexpr (G == 16) x += dpp_move_f64<dpp::kRowMirror>(x);
    return x;
}

// ell_0 .. ell_{N-1} from kappa by one wave: ell_n = -2 sum_{k=1..n} kappa_k
// ell_{n-k}.  The first min(N, 64) pushed forward as each becomes known (lane l
// sums for n = l); the second 64 of N = 128 by one Newton step of the power
// series ell = 1 / h, h = 1 + 2 kappa: r_k = sum_j h_{k-j} ell_j (k = 64..127, j
// < 64), ell_{64+i} = -sum_{j<=i} ell_j r_{64+i-j}: two products of 64 terms per
// lane instead of 64 dependent steps.  kap[-128 .. -1] and kap[0] (kappa_0 :=
// 0) hold zeros; tmp: 128 doubles.
__device__ __forceinline__ void toeplitz_inverse(int N, const double *kap, double *ell, double *tmp, int lane) {
    double acc = 0.0;
    auto bcast = [](double x, int l) {
        const uint64_t b = __builtin_bit_cast(uint64_t, x);
        const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, l);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
        return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
    };
    const double *k0 = kap + lane;
#pragma unroll 8
    for (int m = 0; m < min(N, 64); ++m) {
        const double e = m == 0 ? 1.0 : -2.0 * bcast(acc, m);
        if (lane == 0) ell[m] = e;
        acc = fma(k0[-m], e, acc);
    }
    if (N <= 64) return;
    wave_lds_sync();
    double r[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int j = 0; j < 64; j += 4)
#pragma unroll
        for (int q = 0; q < 4; ++q) r[q] = fma(kap[64 + lane - j - q], ell[j + q], r[q]);
    tmp[lane] = 0.0;
    tmp[64 + lane] = 2.0 * ((r[0] + r[1]) + (r[2] + r[3]));  // r_{64+lane}; zeros below
    wave_lds_sync();
    double a[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int j = 0; j < 64; j += 4)
#pragma unroll
        for (int q = 0; q < 4; ++q) a[q] = fma(ell[j + q], tmp[64 + lane - j - q], a[q]);
    ell[64 + lane] = -((a[0] + a[1]) + (a[2] + a[3]));
}

// One workgroup's entries of A^L.  From e_j the projections of tokens 1..L are
// q_s(j) u_j with q_s = lambda_j q_{s-1} + ell_{s-1}, so (A^L)_ij = delta_ij
// lambda_i^L - 2 u_i u_j sum_s lambda_i^{L-s+1} q_s(j): L independent-entry
// steps in double once ell_0 .. ell_{L-1} are known (kappa_n from tables of
// lambda^0..15 and u^2 lambda^{16 a}).  lds: SegCfg<D>::kLds bytes.
template <int D>
__device__ __forceinline__ void power_entries(int L, const float *lambda, const float *u, float *AL, int wg, char *lds,
                                              double *kap, double *ell) {  // kap[256], ell[128]
    using K = SegCfg<D>;
    constexpr int TS = D + 2;  // padded row of the tables: 24 rows
    static_assert(24 * TS * 8 + K::NT * 8 <= K::kLds && K::NT >= 128, "tables fit the scan's LDS");
    double *t1 = reinterpret_cast<double *>(lds), *t2 = t1 + 16 * TS, *part = t2 + 8 * TS;
    const int tid = threadIdx.x;
    if (tid < D) {
        const double l = lambda[tid], uu = (double)u[tid] * u[tid];
        double x = 1.0;
#pragma unroll
        for (int n = 0; n < 16; ++n) {
            t1[n * TS + tid] = x;
            x *= l;
        }
        double y = uu;
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            t2[n * TS + tid] = y;
            y *= x;
        }
    }
    if (tid < 128) kap[tid] = 0.0;
    __syncthreads();
    {
        constexpr int G = K::NT / 128;  // channel blocks
        const int n = tid & 127, g = tid >> 7;
        double s = 0.0;
        double s4[4] = {0.0, 0.0, 0.0, 0.0};
        for (int c = g * (D / G); c < (g + 1) * (D / G); c += 4)
#pragma unroll
            for (int q = 0; q < 4; ++q) s4[q] = fma(t1[(n & 15) * TS + c + q], t2[(n >> 4) * TS + c + q], s4[q]);
        s = (s4[0] + s4[1]) + (s4[2] + s4[3]);
        part[tid] = s;
        __syncthreads();
        if (tid < 128) {
#pragma unroll
            for (int q = 1; q < G; ++q) s += part[tid + 128 * q];
            kap[128 + tid] = tid == 0 ? 0.0 : s;
        }
    }
    __syncthreads();
    if (tid < 64) toeplitz_inverse(L, kap + 128, ell, part, tid);
    __syncthreads();
    constexpr int E = K::kPowEntries;
    const int idx = wg * K::NT + tid, j = idx % D, i0 = idx / D * E;  // rows i0 .. i0 + E - 1 of column j
    double li[E], acc[E], q = 0.0;
    const double lj = lambda[j];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        li[e] = lambda[i0 + e];
        acc[e] = 0.0;
    }
#pragma unroll 4
    for (int s = 0; s < L; ++s) {
        q = fma(lj, q, ell[s]);
#pragma unroll
        for (int e = 0; e < E; ++e) acc[e] = li[e] * (acc[e] + q);
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
        double pw = li[e];
        for (int n = 1; n < L; n *= 2) pw *= pw;
        const double uu = (double)u[i0 + e] * u[j];
        AL[(size_t)(i0 + e) * D + j] = (float)((i0 + e == j ? pw : 0.0) - 2.0 * uu * acc[e]);
    }
}

template <int D>
__global__ void __launch_bounds__(SegCfg<D>::NT) rosa_power_kernel(int L, const float *lambda, const float *u, float *AL) {
    __shared__ __attribute__((aligned(16))) char lds[SegCfg<D>::kLds];
    __shared__ double kap[256], ell[128];
    power_entries<D>(L, lambda, u, AL, blockIdx.x, lds, kap, ell);
}

// EMIT = false, the first launch: workgroups (chain, segment 0 .. P - 2), then
// those of A^L.  EMIT = true: workgroups (chain, segment).
template <int D, bool EMIT>
__global__ void __launch_bounds__(SegCfg<D>::NT) rosa_seg_kernel(RosaSegParams p) {
    using K = SegCfg<D>;
    constexpr int NT = K::NT, GL = K::GL, PS = K::PS, IT = K::IT, C = kSegC;
    constexpr int KB = D == 256 ? 8 : 16;  // values a chain thread reads ahead
    __shared__ __attribute__((aligned(16))) char lds[K::kLds];
    __shared__ double kap[256], ell[128];
    __shared__ double fv[C + 2], pl[2];  // f_1 .. f_33 (fv[t]); p_33 of the last chunk
    __shared__ __attribute__((aligned(16))) float pn[C + 2];  // -2 p_1 .. -2 p_33 (pn[t])
    __shared__ __attribute__((aligned(16))) float st[2][D];
    __shared__ float part[K::H][D];
    double *prod = reinterpret_cast<double *>(lds);                   // [C][PS]
    float *es = reinterpret_cast<float *>(lds + (size_t)C * PS * 8);  // [C][D]
    float *gs = es + C * D;

    const int tid = threadIdx.x;
    const int segs = EMIT ? p.P : p.P - 1;
    if (!EMIT && (int)blockIdx.x >= p.B * segs) {
        power_entries<D>(p.L, p.lam, p.u, p.AL_out, (int)blockIdx.x - p.B * segs, lds, kap, ell);
        return;
    }
    const int b = blockIdx.x / segs, s = blockIdx.x - b * segs;
    const int t_begin = s * p.L, t_end = min(p.T, t_begin + p.L);
    const bool gated = p.read_raw != nullptr;
    const int slot = p.slot ? p.slot[b] : b;

    // Threads D .. NT - 1: this chunk's raw inputs, and e and the gates made of them.
    const int ct = tid - D;
    float4 in0[IT], in1[IT], in2[IT];
    auto load_in = [&](int t0) {
        const int nt = min(C, t_end - t0);
        const size_t base = ((size_t)b * p.T + t0) * p.ld;
        const uint32_t bytes = (uint32_t)(((nt - 1) * p.ld + D) * 4);
        const auto r0 = make_rsrc(p.cand + base, bytes), r1 = make_rsrc(p.write + base, bytes);
        const auto r2 = make_rsrc(EMIT && gated ? p.read_raw + base : p.cand + base, EMIT && gated ? bytes : 0u);
        int c0 = ct;
        asm volatile("" : "+v"(c0));  // the offsets are formed here: kept over the loop they cost registers (a spill at D = 256)
#pragma unroll
        for (int i = 0; i < IT; ++i) {
            const int q = c0 + i * K::CT, tau = q / (D / 4), c = 4 * (q % (D / 4));
            const uint32_t off = tau < nt && c0 >= 0 ? (uint32_t)(tau * p.ld + c) * 4u : kBufferOob;
            in0[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r0, off, 0, 0));
            in1[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r1, off, 0, 0));
            if constexpr (EMIT) in2[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r2, off, 0, 0));
        }
    };
    auto make_e = [&]() {  // in0 <- e (out-of-range tokens read 0 and give 0)
#pragma unroll
        for (int i = 0; i < IT; ++i)
            in0[i] = make_float4(seg_cand(in0[i].x, in1[i].x), seg_cand(in0[i].y, in1[i].y),
                                 seg_cand(in0[i].z, in1[i].z), seg_cand(in0[i].w, in1[i].w));
    };
    auto make_gates = [&]() {
        if constexpr (EMIT)
            if (gated)
#pragma unroll
                for (int i = 0; i < IT; ++i)
                    in2[i] = make_float4(seg_gate(in2[i].x), seg_gate(in2[i].y), seg_gate(in2[i].z), seg_gate(in2[i].w));
    };
    auto stage = [&]() {  // e and the gates to LDS
#pragma unroll
        for (int i = 0; i < IT; ++i) {
            const int q = ct + i * K::CT;
            if (q < C * D / 4) {
                reinterpret_cast<float4 *>(es)[q] = in0[i];
                if constexpr (EMIT) reinterpret_cast<float4 *>(gs)[q] = in2[i];
            }
        }
    };
    const bool chain = tid < D;
    // Loaded ahead of everything, except that at D = 256 the carry's A^L rows
    // (128 registers) leave no room for a chunk's inputs beside them.
    const bool walk = EMIT && p.P > 1 && !p.starts && s > 1;
    if (!chain && !(D == 256 && walk)) load_in(t_begin);

    // Start state: the chain's own, zero, or A^L walked over the segments before.
    const float lam = tid < D ? p.lam[tid] : 0.0f, u = tid < D ? p.u[tid] : 0.0f;
    float m = 0.0f;
    if constexpr (!EMIT) {
        if (s == 0 && tid < D) {
            m = p.memory_in ? p.memory_in[(size_t)slot * D + tid] : 0.0f;
            p.z[((size_t)b * p.P + p.P - 1) * D + tid] = m;
        }
    } else if (p.P == 1) {
        if (tid < D && p.memory_in) m = p.memory_in[(size_t)slot * D + tid];
    } else if (p.starts) {
        if (tid < D) m = p.starts[((size_t)b * p.P + s) * D + tid];
    } else {
        if (tid < D) m = p.z[((size_t)b * p.P + (s == 0 ? p.P - 1 : 0)) * D + tid];
    }

    const int tau = tid / GL, gl = tid % GL;
    auto dot_row = [&]() {  // sum of row tau of prod, to the GL lanes of its group
        double a0 = 0.0, a1 = 0.0;
        typedef double doublex2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int i = 0; i < D / (2 * GL); ++i) {
            const doublex2 v = *reinterpret_cast<const doublex2 *>(prod + tau * PS + 2 * (gl + GL * i));
            a0 += v[0];
            a1 += v[1];
        }
        return group_sum_f64<GL>(a0 + a1);
    };
    // ell_0 .. ell_32 of a chunk, kept by the first launch for the second.
    if (EMIT && p.P > 1) {
        if (tid < C + 1) ell[tid] = p.ell[(size_t)b * kSegEll + tid];
    } else {
        if (chain) {
            double pw = (double)u * u;
#pragma unroll
            for (int n = 0; n < C; ++n) {
                pw *= lam;
                prod[n * PS + tid] = pw;
            }
        }
        if (tid < 128) kap[tid] = 0.0;
        if (tid > C && tid < 128) kap[128 + tid] = 0.0;
        if (tid == 0) kap[128] = 0.0;
        lds_barrier();
        const double k = dot_row();
        if (gl == 0) kap[128 + tau + 1] = k;
        lds_barrier();
        if (tid < 64) {
            toeplitz_inverse(C + 1, kap + 128, ell, kap, tid);
            if (!EMIT && s == 0) {
                wave_lds_sync();
                if (tid < C + 1) p.ell[(size_t)b * kSegEll + tid] = ell[tid];
            }
        }
    }

    if constexpr (EMIT) {
        if (walk) {  // uniform over the workgroup
            constexpr int W = K::W, H = K::H;
            const int r = tid % D, h = tid / D;
            float arow[W];
            const float4 *a4 = reinterpret_cast<const float4 *>(p.AL + (size_t)r * D + h * W);
#pragma unroll
            for (int j = 0; j < W / 4; ++j) {
                const float4 t = a4[j];
                arow[4 * j] = t.x; arow[4 * j + 1] = t.y; arow[4 * j + 2] = t.z; arow[4 * j + 3] = t.w;
            }
            const float *zr = p.z + (size_t)b * p.P * D;
            if (tid < D) st[0][tid] = m;
            float zn = tid < D ? zr[D + tid] : 0.0f;
            lds_barrier();
            for (int j = 1; j < s; ++j) {
                const float4 *x4 = reinterpret_cast<const float4 *>(st[(j - 1) & 1] + h * W);
                float d4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int q = 0; q < W / 4; ++q) {
                    const float4 x = x4[q];
                    d4[0] = fmaf(arow[4 * q], x.x, d4[0]);
                    d4[1] = fmaf(arow[4 * q + 1], x.y, d4[1]);
                    d4[2] = fmaf(arow[4 * q + 2], x.z, d4[2]);
                    d4[3] = fmaf(arow[4 * q + 3], x.w, d4[3]);
                    if (D == 256 && q % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // 16 state values at a time in registers
                }
                part[h][r] = (d4[0] + d4[1]) + (d4[2] + d4[3]);
                const float zj = zn;
                if (tid < D && j + 1 < s) zn = zr[(size_t)(j + 1) * D + tid];
                lds_barrier();
                if (tid < D) {
                    float sum = part[0][tid];
#pragma unroll
                    for (int q = 1; q < H; ++q) sum += part[q][tid];
                    m = sum + zj;
                    st[j & 1][tid] = m;
                }
                lds_barrier();
            }
            if (D == 256) load_in(t_begin);  // by every thread (a chain thread reads nothing): no value is kept across the walk
        }
    }

    // f_1 = u.m of the first chunk: row 0 of prod.
    lds_barrier();
    if (chain) {
        prod[tid] = (double)u * (double)m;
    } else {
        make_e();
        make_gates();
        stage();
        if (t_begin + C < t_end) load_in(t_begin + C);
    }
    lds_barrier();
    {
        const double f = dot_row();  // rows above 0: unused
        if (tid == 0) fv[1] = f;
    }
    lds_barrier();

    for (int t0 = t_begin; t0 < t_end; t0 += C) {
        const int nt = min(C, t_end - t0);
        const bool more = t0 + C < t_end;
        if (chain) {
            double y = m;
            const double ld = lam, ud = u;
            // A block of values ahead of the stores: those may alias the reads to the
            // compiler, and a read behind each would put its latency in the chain.
#pragma unroll
            for (int k0 = 0; k0 < C; k0 += KB) {
                float ev[KB];
#pragma unroll
                for (int k = 0; k < KB; ++k) ev[k] = es[(k0 + k) * D + tid];
#pragma unroll
                for (int k = 0; k < KB; ++k) {
                    y = fma(ld, y, (double)ev[k]);
                    prod[(k0 + k) * PS + tid] = ud * y;
                }
            }
        } else if (more) {
            make_e();
        }
        lds_barrier();
        {
            const double f = dot_row();
            if (gl == 0) fv[tau + 2] = f;
        }
        lds_barrier();
        {
            // p_t = sum_{q=1..t} ell_{t-q} f_q, t = tau + 2.
            const int t = tau + 2;
            double a = 0.0;
#pragma unroll
            for (int i = 0; i < (C + 1 + GL - 1) / GL; ++i) {
                const int q = 1 + gl + GL * i;
                a = fma(q <= t ? ell[q <= t ? t - q : 0] : 0.0, q <= t ? fv[q <= t ? q : 1] : 0.0, a);
            }
            a = group_sum_f64<GL>(a);
            if (gl == 0) pn[t] = (float)(-2.0 * a);
            if (tid == 0) pn[1] = (float)(-2.0 * fv[1]);
            if (tau == C - 1 && gl == 0) pl[0] = a;
        }
        lds_barrier();
        if (chain) {
            if (tid == 0) fv[1] = pl[0];  // p_33; read again only behind the next chunk's barriers
            float *out = EMIT ? p.read_out + ((size_t)b * p.T + t0) * D + tid : nullptr;
            auto run = [&](int n) {
#pragma unroll
                for (int k0 = 0; k0 < C; k0 += KB) {
                    float ev[KB], gv[KB], pv[KB + 1];
#pragma unroll
                    for (int k = 0; k < KB; ++k) {
                        ev[k] = es[(k0 + k) * D + tid];
                        gv[k] = EMIT && gated ? gs[(k0 + k) * D + tid] : 1.0f;
                        pv[k] = pn[k0 + k + 1];
                    }
                    pv[KB] = pn[k0 + KB + 1];
#pragma unroll
                    for (int k = 0; k < KB; ++k) {
                        if (k0 + k >= n) break;
                        m = fmaf(lam, fmaf(pv[k], u, m), ev[k]);
                        if constexpr (EMIT) out[(size_t)(k0 + k) * D] = fmaf(pv[k + 1], u, m) * gv[k];
                    }
                }
            };
            if (nt == C) run(C);
            else run(nt);
        } else if (more) {
            make_gates();
        }
        lds_barrier();
        if (!chain && more) {
            stage();
            if (t0 + 2 * C < t_end) load_in(t0 + 2 * C);
        }
        lds_barrier();
    }
    if (tid < D) {
        if constexpr (!EMIT) p.z[((size_t)b * p.P + s) * D + tid] = m;
        else if (p.memory_out && s == p.P - 1) p.memory_out[(size_t)slot * D + tid] = m;
    }
}

template <int D>
hipError_t launch_power(int L, const float *lambda, const float *u, float *AL, hipStream_t stream) {
    hipLaunchKernelGGL(rosa_power_kernel<D>, dim3(SegCfg<D>::kPowWgs), dim3(SegCfg<D>::NT), 0, stream, L, lambda, u, AL);
    return hipGetLastError();
}

hipError_t launch_rosa_power(int D, int L, const float *lambda, const float *u, float *AL, hipStream_t stream) {
    if (L < 1 || L > 128 || (L & (L - 1)) != 0) return hipErrorInvalidValue;
    if (D == 64) return launch_power<64>(L, lambda, u, AL, stream);
    if (D == 128) return launch_power<128>(L, lambda, u, AL, stream);
    if (D == 256) return launch_power<256>(L, lambda, u, AL, stream);
    return hipErrorInvalidValue;
}

bool rosa_seg_ok(int T, int D) { return T > 1 && (D == 64 || D == 128 || D == 256); }

// One segment up to 192 tokens (the longer chain costs what a second launch
// does: 22 against 21 us at D = 128, 35 / 33 at D = 256), then 64-token segments
// (8 x 640 x 128: 24 us, 31 with 128-token ones), and 128-token segments where the
// carry and the workgroups of 64-token ones cost more (8 x 4096 x 128: 46 against
// 64; 32 x 1111: 51 / 61 but 1 x 1111: 32 / 27).  By length alone, so that a
// batch's parts are cut like the whole.
int rosa_seg_len(int T) { return T < 1024 ? 64 : 128; }
int rosa_segments(int T) { return T <= 192 ? 1 : (T + rosa_seg_len(T) - 1) / rosa_seg_len(T); }

size_t rosa_seg_scratch(int B, int T, int D) {
    const int P = rosa_segments(T);
    return P == 1 ? 0 : (size_t)B * (2 * P * D + (P > kRosaChain ? 2 * kSegEll : 0));
}

template <int D>
hipError_t launch_seg(RosaSegParams q, float *carry, hipStream_t stream) {
    const dim3 block(SegCfg<D>::NT);
    hipError_t e = hipSuccess;
    if (q.P > 1) {
        const unsigned extra = q.AL_out ? SegCfg<D>::kPowWgs : 0;
        hipLaunchKernelGGL((rosa_seg_kernel<D, false>), dim3((unsigned)(q.B * (q.P - 1)) + extra), block, 0, stream, q);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        if (q.P > kRosaChain) {
            hipLaunchKernelGGL(rosa_carry_kernel<D>, dim3(q.B), dim3(D * D / 64), 0, stream, q.P, q.AL, q.z, carry);
            if ((e = hipGetLastError()) != hipSuccess) return e;
            q.starts = carry;
        }
    }
    hipLaunchKernelGGL((rosa_seg_kernel<D, true>), dim3((unsigned)(q.B * q.P)), block, 0, stream, q);
    return hipGetLastError();
}

hipError_t launch_rosa_segmented(const RosaParams &p, const float *AL, float *scratch, hipStream_t stream) {
    if (p.B <= 0) return hipSuccess;
    if (!rosa_seg_ok(p.T, p.D) || p.raw_params || !p.cand || !p.write || !p.read_out) return hipErrorInvalidValue;
    RosaSegParams q;
    q.B = p.B; q.T = p.T; q.ld = p.ld; q.L = rosa_seg_len(p.T); q.P = scratch ? rosa_segments(p.T) : 1;
    q.cand = p.cand; q.write = p.write; q.read_raw = p.read_raw;
    q.lam = p.decay; q.u = p.direction;
    q.memory_in = p.memory_in; q.memory_out = p.memory_out; q.slot = p.slot; q.read_out = p.read_out;
    float *carry = nullptr;
    if (q.P > 1) {
        // z, then the carry pass's start states -- ell where there is no such
        // pass, else ell after them -- then A^L if it is not given.
        const size_t rows = (size_t)p.B * q.P * p.D;
        q.z = scratch;
        carry = scratch + rows;
        q.ell = reinterpret_cast<double *>(q.P > kRosaChain ? carry + rows : carry);
        q.AL = AL;
        if (!AL) q.AL = q.AL_out = scratch + rosa_seg_scratch(p.B, p.T, p.D);
    } else {
        q.L = p.T;
    }
    if (p.D == 64) return launch_seg<64>(q, carry, stream);
    if (p.D == 128) return launch_seg<128>(q, carry, stream);
    return launch_seg<256>(q, carry, stream);
}

namespace {
// Operator path: scratch of the segmented scan, one growing buffer per (device,
// stream) kept for the life of the process.  A stream's launches wait on its
// earlier ones, so its calls can share a buffer if the launches of one call
// follow each other: g_rosa_mu is held from the choice of the buffer to the
// call's last launch.  The handle of the per-thread default stream stands for
// another stream in each thread.  An outgrown buffer is not freed, since launches
// in flight or a captured graph may still use it; the next one is at least twice
// as large, so what a stream has outgrown is less than what it uses.  Calls under
// capture have a buffer apart from the stream's eager calls, beside which the
// graph may be replayed.
using RosaScratchKey = std::tuple<int, hipStream_t, std::thread::id, bool>;
std::mutex g_rosa_mu;
std::map<RosaScratchKey, std::pair<float *, size_t>> g_rosa_scratch;

bool op_rosa_sequential() {
    const char *e = std::getenv("YUF_ROSA_SEGMENTED");
    return e && std::strcmp(e, "0") == 0;
}

// With g_rosa_mu held.
hipError_t op_rosa_scratch(hipStream_t stream, bool capturing, size_t floats, float **out) {
    int dev = 0;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return err;
    const std::thread::id owner = stream == hipStreamPerThread ? std::this_thread::get_id() : std::thread::id();
    auto &slot = g_rosa_scratch[{dev, stream, owner, capturing}];
    if (slot.second < floats) {
        const size_t size = std::max(floats, 2 * slot.second);
        // Allocating is no stream operation: it may happen while this or another stream is captured.
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        if ((err = hipThreadExchangeStreamCaptureMode(&mode)) != hipSuccess) return err;
        float *p = nullptr;
        err = hipMalloc(&p, size * sizeof(float));
        const hipError_t back = hipThreadExchangeStreamCaptureMode(&mode);
        if (err != hipSuccess) return err;
        slot = {p, size};
        if (back != hipSuccess) return back;
    }
    *out = slot.first;
    return hipSuccess;
}
}  // namespace

hipError_t launch_rosa(const RosaParams &p, hipStream_t stream) {
    if (p.B <= 0) return hipSuccess;
    if (p.T == 1) {
        const dim3 grid((p.B + 3) / 4), block(256);
        const int epl = (p.D + kWave - 1) / kWave;
        if (epl <= 1) hipLaunchKernelGGL(rosa_step_kernel<1>, grid, block, 0, stream, p);
        else if (epl <= 2) hipLaunchKernelGGL(rosa_step_kernel<2>, grid, block, 0, stream, p);
        else if (epl <= 4) hipLaunchKernelGGL(rosa_step_kernel<4>, grid, block, 0, stream, p);
        else if (epl <= 8) hipLaunchKernelGGL(rosa_step_kernel<8>, grid, block, 0, stream, p);
        else if (epl <= 16) hipLaunchKernelGGL(rosa_step_kernel<16>, grid, block, 0, stream, p);
        else return hipErrorInvalidValue;
        return hipGetLastError();
    }
    const dim3 grid(p.B), block(kThreads);
    const int epl = (p.D + kWave - 1) / kWave;
    if (epl <= 1) hipLaunchKernelGGL(rosa_scan_kernel<1>, grid, block, 0, stream, p);
    else if (epl <= 2) hipLaunchKernelGGL(rosa_scan_kernel<2>, grid, block, 0, stream, p);
    else if (epl <= 4) hipLaunchKernelGGL(rosa_scan_kernel<4>, grid, block, 0, stream, p);
    else if (epl <= 8) hipLaunchKernelGGL(rosa_scan_kernel<8>, grid, block, 0, stream, p);
    else if (epl <= 16) hipLaunchKernelGGL(rosa_scan_kernel<16>, grid, block, 0, stream, p);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace yuf

namespace yuf {
namespace {

// The no-allocation operator variant (yuf_rosa_scan_f32_noalloc) keeps the
// segmented scan's scratch -- A^L and the z / carry segment rows -- in
// this file-scope device array: every device the library runs on holds one
// copy, at its own address, until the process ends.  Nothing in it needs to
// start at zero (each pass writes its rows before the next reads them).
constexpr size_t kNoAllocScratchFloats = (size_t)4 << 20;  // 16 MiB
__device__ __align__(256) float scratch[kNoAllocScratchFloats];

// Device address of `scratch` per device, resolved once per device with that
// device current (the array's name is a host-side stand-in, never passed to a
// kernel).  Fixed storage: no host or device allocation on this path.
constexpr int kNoAllocMaxDevices = 64;
std::mutex g_noalloc_mu;
float *g_noalloc_ptr[kNoAllocMaxDevices] = {};

int noalloc_scratch(float **out) {
    int dev = 0;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return fail(YUF_ERR_HIP, std::string("rosa noalloc: hipGetDevice: ") + hipGetErrorString(err));
    if (dev < 0 || dev >= kNoAllocMaxDevices) return fail(YUF_ERR_INVALID, "rosa noalloc: device index above 63");
    std::lock_guard<std::mutex> lock(g_noalloc_mu);
    if (!g_noalloc_ptr[dev]) {
        void *ptr = nullptr;
        err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (err != hipSuccess || !ptr)
            return fail(YUF_ERR_HIP, std::string("rosa noalloc: hipGetSymbolAddress: ") + hipGetErrorString(err));
        g_noalloc_ptr[dev] = static_cast<float *>(ptr);
    }
    *out = g_noalloc_ptr[dev];
    return YUF_OK;
}

// The operator: argument checks, then the segment form (scratch from the growing
// per-stream buffer, or from `scratch` when noalloc; none for one segment) or,
// for other D, the sequential chunked scan (no scratch).  The no-allocation
// variant does not read YUF_ROSA_SEGMENTED: its scratch capacity is checked on
// every multiple of 64 that can take segments, before any launch, whatever the
// switch says.
int rosa_operator(int B, int T, int D, const float *cand, const float *write, const float *read_raw,
                  const float *decay, const float *direction, const float *memory_in, float *memory_out,
                  float *read_out, void *stream, bool noalloc) {
    if (B < 0 || T < 0) return fail(YUF_ERR_INVALID, "rosa: negative size");
    if (D < 1 || D > 1024) return fail(YUF_ERR_INVALID, "rosa: D must be in [1, 1024], got " + std::to_string(D));
    if (!decay || !direction) return fail(YUF_ERR_INVALID, "rosa: null decay/direction");
    if (T > 0 && (!cand || !write || !read_out)) return fail(YUF_ERR_INVALID, "rosa: null input/output pointer");
    RosaParams p;
    p.B = B; p.T = T; p.D = D; p.ld = D;
    p.cand = cand; p.write = write; p.read_raw = read_raw;
    p.decay = decay; p.direction = direction;
    p.memory_in = memory_in; p.memory_out = memory_out; p.read_out = read_out;
    const hipStream_t st = static_cast<hipStream_t>(stream);
    hipError_t err = hipSuccess;
    // Shapes that the no-allocation entry point refuses above its documented
    // capacity (64-token segments: never less than what the call uses).
    const bool bounded = B > 0 && T >= 128 && T % 64 == 0 && (D == 64 || D == 128 || D == 256);
    if (noalloc && bounded) {
        const size_t seg = (size_t)B * (T / 64) * D, need = (size_t)D * D + 2 * seg;
        if (need > kNoAllocScratchFloats)
            return fail(YUF_ERR_INVALID, "rosa noalloc: B * (T / 64) * D = " + std::to_string(seg) +
                                             " needs " + std::to_string(need) + " scratch floats (D^2 + 2 B (T / 64) D); "
                                             "the static buffer holds " + std::to_string(kNoAllocScratchFloats) +
                                             " -- split the batch or use yuf_rosa_scan_f32");
    }
    // Up to 8 tokens of D = 256 are two of the sequential scan's chunks (8.2 us,
    // 9.9 as one 32-token chunk; 9 tokens 10.7 / 10.1; the engine, which would launch
    // the gates apart for it, keeps the segment kernel).
    const bool few = D == 256 && T <= 8;
    if (B <= 0 || T <= 0 || !rosa_seg_ok(T, D) || few || (!noalloc && op_rosa_sequential())) {
        err = launch_rosa(p, st);
    } else {
        // Segments (as the engine's prefill), or one segment, which needs no
        // scratch: for ragged lengths under capture (graphs of them may be
        // replayed beside each other; graphs of multiples of 64 share their
        // capture stream's buffer), for ragged lengths of the no-allocation entry
        // point that its array does not hold, and where the buffer cannot be had.
        float *buf = nullptr;
        std::unique_lock<std::mutex> lock(g_rosa_mu, std::defer_lock);
        const size_t need = rosa_seg_scratch(B, T, D) + (size_t)D * D;
        if (rosa_segments(T) > 1 && noalloc) {
            if (bounded || need <= kNoAllocScratchFloats) {
                int rc = noalloc_scratch(&buf);
                if (rc != YUF_OK) return rc;
            }
        } else if (rosa_segments(T) > 1) {
            hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
            const bool known = hipStreamIsCapturing(st, &cap) == hipSuccess;
            const bool capturing = cap != hipStreamCaptureStatusNone;
            lock.lock();
            if (!known || (capturing && !bounded) ||
                op_rosa_scratch(st, capturing, need, &buf) != hipSuccess)
                buf = nullptr;
            if (!buf) (void)hipGetLastError();
        }
        err = launch_rosa_segmented(p, nullptr, buf, st);
    }
    if (err != hipSuccess) return fail(YUF_ERR_HIP, std::string("rosa launch: ") + hipGetErrorString(err));
    return YUF_OK;
}

}  // namespace
}  // namespace yuf

extern "C" int yuf_rosa_scan_f32(int B, int T, int D, const float *cand, const float *write,
                                 const float *read_raw, const float *decay, const float *direction,
                                 const float *memory_in, float *memory_out, float *read_out, void *stream) {
    return yuf::rosa_operator(B, T, D, cand, write, read_raw, decay, direction, memory_in, memory_out, read_out,
                              stream, false);
}

extern "C" int yuf_rosa_scan_f32_noalloc(int B, int T, int D, const float *cand, const float *write,
                                         const float *read_raw, const float *decay, const float *direction,
                                         const float *memory_in, float *memory_out, float *read_out, void *stream) {
    return yuf::rosa_operator(B, T, D, cand, write, read_raw, decay, direction, memory_in, memory_out, read_out,
                              stream, true);
}
