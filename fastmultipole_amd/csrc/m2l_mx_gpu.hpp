// Matrix-core M2L on gfx950: the backend of the engine in m2l_mx.hpp for one wavefront and its
// persistent launch. Included by one translation unit per order cap (m2l_mx_c*.hip), so the caps
// compile in parallel.
#pragma once
#include "expansions_common.hpp"
#include "m2l_mx.hpp"
#include <algorithm>
#include <climits>
#include <cstddef>
#include <cstdlib>

namespace fmmhip {

// ================================ M2L on matrix cores, register-resident (m2l_mx.hpp)
// Backend of the engine in m2l_mx.hpp for one gfx950 wavefront: a per-lane value is a register,
// neighbouring lanes are read with DPP (quad permutations, row rotations), other lanes with
// ds_bpermute (__shfl), and the product is v_mfma_f64_4x4x4_4b_f64.
template <int CTRL>
__device__ __forceinline__ double dpp_d(double x) {
    const long long u = __double_as_longlong(x);
    // every lane has a source: no old value to keep (with one, each move is preceded by a copy)
    const int lo = __builtin_amdgcn_mov_dpp((int)u, CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(u >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
static constexpr int DPP_QUAD(int a, int b, int c, int d) { return a | (b << 2) | (c << 4) | (d << 6); }
static constexpr int DPP_ROW_ROR(int n) { return 0x120 + n; }

struct MxGpu {
    using V = double;
    using I = int;
    using M = bool;
    using PV = const double*;
    static __device__ __forceinline__ I lane() { return (int)(threadIdx.x & 63); }
    static __device__ __forceinline__ V sel(M m, V a, V b) { return m ? a : b; }
    static __device__ __forceinline__ I seli(M m, I a, I b) { return m ? a : b; }
    static __device__ __forceinline__ I mini(I a, int b) { return min(a, b); }
    static __device__ __forceinline__ void sched_fence() { __builtin_amdgcn_sched_barrier(0); }
    static __device__ __forceinline__ I opaque(I a) {   // a value the compiler cannot move out of its scope
        asm volatile("" : "+v"(a));
        return a;
    }
    static __device__ __forceinline__ V fabs(V a) { return ::fabs(a); }
    static __device__ __forceinline__ V sqrt(V a) { return ::sqrt(a); }
    static __device__ __forceinline__ V fma(V a, V b, V c) { return ::fma(a, b, c); }
    static __device__ __forceinline__ V tod(I a) { return (double)a; }
    static __device__ __forceinline__ V perm1(V a) { return dpp_d<DPP_QUAD(1, 0, 3, 2)>(a); }
    static __device__ __forceinline__ V bperm(V a, I src) { return __shfl(a, src, 64); }
    static __device__ __forceinline__ V quadsum(V a) {
        const V b = a + __shfl_xor(a, 16, 64);
        return b + __shfl_xor(b, 32, 64);
    }
    template <int NC>
    static __device__ __forceinline__ V slotsum(V a) {   // sum over lanes of the row with the same lane % NC
        V b = a + dpp_d<DPP_ROW_ROR(8)>(a);
        b = b + dpp_d<DPP_ROW_ROR(4)>(b);
        b = b + dpp_d<DPP_ROW_ROR(2)>(b);
        if constexpr (NC == 1) b = b + dpp_d<DPP_ROW_ROR(1)>(b);
        return b;
    }
    template <int NC, int j>
    static __device__ __forceinline__ V qbcast(V a) {   // of columns NC i + (0 .. NC - 1), the value of column NC i + j
        static_assert(NC == 2, "columns come in pairs");
        return dpp_d<DPP_QUAD(j, j, 2 + j, 2 + j)>(a);
    }
    static __device__ __forceinline__ V mfma4(V a, V b, V d) { return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, d, 0, 0, 0); }
    static __device__ __forceinline__ bool any(M m) { return __ballot(m) != 0ull; }
    static __device__ __forceinline__ bool all(M m) { return __ballot(!m) == 0ull; }
    static __device__ __forceinline__ int maxi(I a, M m) {
        int v = m ? a : INT_MIN;
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
        return v;
    }
    static __device__ __forceinline__ V gld(const double* p, I i, M ok) {
        V r = 0.0;
        if (ok) r = p[i];
        return r;
    }
    static __device__ __forceinline__ I gldi(const int32_t* p, I i, M ok) {
        I r = 0;
        if (ok) r = p[i];
        return r;
    }
    static __device__ __forceinline__ PV ptr(const double* base, I js, int64_t stride) { return base + (int64_t)js * stride; }
    static __device__ __forceinline__ V gldp(PV p, I i) { return p[i]; }
    static __device__ __forceinline__ V lds(const double* p, I i) { return p[i]; }
    static __device__ __forceinline__ void lds_st(double* p, I i, V x, M ok) {
        if (ok) p[i] = x;
    }
    static __device__ __forceinline__ void lds_add(double* p, I i, V x, M ok) {
        if (ok) p[i] += x;
    }
    static __device__ __forceinline__ void sti(int32_t* p, I i, I x, M ok) {
        if (ok) p[i] = x;
    }
    static __device__ __forceinline__ void wsync() { wave_sync(); }
};

template <int CAP, bool LH>
static size_t mx_lds_bytes(int nw) {
    return sizeof(double) * (size_t)(mx::shared_doubles<CAP>() + nw * mx::wave_doubles<CAP, LH>());
}

// Work items. A target box's list entries are cut into chunks of S (the last one shorter), and a wavefront takes one
// chunk at a time: with a wavefront per box the launch lasted as long as its longest list (45k ring at cap 20, 24,644
// interactions in 1,400 boxes: 4.05 ms; 0.8 ms in chunks). Chunk c of
// box b has slot l0 / S + b + c, l0 the box's first list entry: chunks of different boxes never share a slot
// (ceil(len / S) <= floor(l1 / S) - floor(l0 / S) + 1), and the last slot is known on the host without a scan.
// A box of one chunk is added to its target's expansion by the wavefront that holds it; the chunks of the others go to
// `part` and k_m2l_mx_sum adds them in chunk order. S depends on the cap alone, never on the size of the problem, so a
// box's sum is the same to the last bit whatever is evaluated beside it. S is one batch up to cap 12 and two above: a
// chunk's partial expansion (7.4 KB at cap 20) is written and read once per S interactions, 1.2 GB of the 1M ring's 32 GB.
__host__ __device__ inline int64_t mx_first_slot(int64_t l0, int64_t box, int S) { return l0 / S + box; }

// The partial expansions take M2L_PART_BYTES at most (or two of the longest lists possible, if that is more: from about 0.6M
// branches at order 20). The slots of larger launches are taken in passes: the pass from w0 to w1 takes every chunk of the
// boxes whose first slot lies in it, up to `span` slots past w1 (a list holds a source branch once, so its chunks are no
// more than n_branches / S), and k_m2l_mx_sum adds them before the next pass. A box is summed
// whole in one pass, so its sum does not depend on where the passes end. One pass for 4M bodies at order 8 (1.1 GB) or
// the 1M ring at order 20 (1.0 GB); without a bound 2.5M uniform vortices at order 20 (37M interactions) took 20.7 GiB,
// and 428 ms against 430 ms in ten passes.

// the box whose slots hold slot w: the last one whose first slot is not above w (64 candidates per step)
__device__ inline int mx_box_of(const int64_t* __restrict__ m2l_offsets, int n_boxes, int64_t w, int S, int lane) {
    int lo = 0, len = n_boxes;
    while (len > 1) {
        const int step = (len + 63) >> 6;
        const int k = lo + (lane + 1) * step;
        const bool below = (lane + 1) * step < len && mx_first_slot(m2l_offsets[k], k, S) <= w;
        const int moves = __popcll(__ballot(below));
        lo += moves * step;
        len = min(step, len - moves * step);
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

// Persistent: every workgroup copies the tables into LDS once, then each wavefront takes chunks, `grab` slots at a time,
// from a counter (flags[2], from 0 in every pass) and runs their interactions BP at a time, summed in the wavefront's LDS.
//
// What bounds it: at cap 8 and 12 two or three wavefronts per SIMD, 40 % of the cycles on the vector ALU and matrix
// cores, the rest waits on LDS and the gathered expansions (4M Plummer sphere, order 8, 22.9M interactions: 31.9 -> 9.0 ms,
// 2.5e9 translations/s). At cap 16 and 20 the local expansion fills the registers (204 and 300 per lane; beyond 256
// they move through accumulation registers), one wavefront per SIMD, LDS latency exposed (300k sphere, order 16:
// 7.6 -> 3.7 ms, 6.3 ms when forced to two wavefronts; 1M ring, orders to 20: 28 -> 20.3 ms). What does not fit 512 registers
// goes to scratch memory: with the tests and two potentials 1.3 KB a lane at cap 20, about 23 of the 32 GB that the 1M
// ring's launch moves, and 0.3 KB at cap 16; 0.1 to 0.6 KB at cap 12, held to 256 for its two wavefronts.
template <int CAP, bool LH, int NW, bool ERR>
__global__ __launch_bounds__(64 * NW, CAP <= 12 ? 2 : 1) void k_m2l_mx(const int32_t* __restrict__ m2l_targets,
                                                    const int64_t* __restrict__ m2l_offsets,
                                                    const int32_t* __restrict__ m2l_s, const Branch* __restrict__ tbr,
                                                    const Branch* __restrict__ sbr, const double* __restrict__ sex,
                                                    double* __restrict__ tex, double* __restrict__ part, int n_boxes,
                                                    int w0, int w1, int wend, int grab, int P, int PE, ErrParams E,
                                                    const int32_t* __restrict__ perm, int32_t* __restrict__ orders,
                                                    int32_t* __restrict__ flags, int32_t* __restrict__ box_ok,
                                                    TablePtrs tb) {
    using Eng = mx::Engine<MxGpu, CAP, LH, ERR>;
    constexpr int H = nh(CAP), NC = Eng::NC, BP = Eng::BP, NS = CAP + 1;
    extern __shared__ double lds[];
    const mx::Tabs T = mx::tabs<CAP>(lds);
#pragma unroll CAP <= 12 ? CAP + 1 : 1
    for (int n = 0, at = 0; n <= CAP; ++n) {
        const int len = 16 * (mx::KE(n) + mx::KO(n)) * (mx::KE(n) + mx::KO(n));
        for (int t = threadIdx.x; t < len; t += blockDim.x) T.A[at + t] = mx::padded(tb.Ad, n, t);
        at += len;
    }
    for (int i = threadIdx.x; i < H; i += blockDim.x) {
        int n, m;
        idx_nm(i, n, m);
        const int b = len_Ts(n - 1);
        T.zin[i] = tb.zeta[b + m];
        T.zoh[i] = 0.5 * tb.zeta[b + m * (n + 1)];
        T.ein[i] = tb.eta[b + m];
        T.eoh[i] = 0.5 * tb.eta[b + m * (n + 1)];
        T.Mt[i] = tb.Mt[i];
        T.Lt[i] = tb.Lt[i];
    }
    for (int i = threadIdx.x; i < 2 * NS; i += blockDim.x) T.tf[i] = tb.tfac[i];
    for (int n = threadIdx.x; n < NS; n += blockDim.x) {
        T.i0[2 * n] = 1.0 / tb.Mt[nh(n - 1)];
        T.i0[2 * n + 1] = 1.0 / tb.Lt[nh(n - 1)];
    }
    __syncthreads();
    const mx::Wave W = mx::wave<CAP, LH>(lds + mx::shared_doubles<CAP>() + (size_t)wave_id() * mx::wave_doubles<CAP, LH>());
    const int64_t HE4 = 4 * (int64_t)nh(PE);
    const int lane = lane_id();
    int pmax = 0, okf = 1;
    constexpr int S = m2l_chunk(CAP, LH);
    int slot = -1, left = 0, box = 0;
    int64_t lb = 0, le = 0;
    for (;;) {
        if (left == 0) {
            if (grab == 0) {   // one slot per wavefront
                if (slot >= 0) break;
                slot = w0 + (int)blockIdx.x * NW + __builtin_amdgcn_readfirstlane(wave_id());
                if (slot >= wend) break;
                left = 1;
            } else {
                if (lane == 0) slot = w0 + atomicAdd(flags + 2, grab);
                slot = __builtin_amdgcn_readfirstlane(slot);
                if (slot >= wend) break;
                left = min(grab, wend - slot);
            }
            box = mx_box_of(m2l_offsets, n_boxes, slot, S, lane);
            lb = m2l_offsets[box];
            le = m2l_offsets[box + 1];
        } else if (box + 1 < n_boxes && mx_first_slot(le, box + 1, S) <= slot) {
            ++box;
            lb = le;
            le = m2l_offsets[box + 1];
        }
        const int first = (int)mx_first_slot(lb, box, S);
        const int64_t l0 = lb + (int64_t)(slot - first) * S, l1 = min(le, l0 + S);
        const int at = slot++ - w0;
        --left;
        if (l0 >= le || first < w0 || first >= w1) continue;   // one chunk fewer than slots, or a box of another pass
        for (int i = lane; i < NC * H; i += 64) W.acc[i] = 0.0;
        wave_sync();
        const int32_t it = m2l_targets[box];
        const Branch& Tb = tbr[it];
        mx::Box X;
        for (int d = 0; d < 3; ++d) {
            X.tc[d] = Tb.target_center[d];
            X.tbox[d] = Tb.target_box[d];
        }
        X.r_l = Tb.target_radius;
        const double eps = E.relative ? Tb.max_influence * E.eps : E.eps;
        X.limit = eps * 4 * PI_D;
        X.P = P;
        X.kind = E.kind;
        X.BE = E.BE;
        int okb = 1;
        for (int64_t b0 = l0; b0 < l1; b0 += BP) {
            const mx::Batch Bt{m2l_s, perm, (int)b0, (int)min((int64_t)BP, l1 - b0), orders};
            Eng::batch(T, W, X, Bt, (const double*)sbr, (int)(sizeof(Branch) / 8), (int)(offsetof(Branch, source_center) / 8),
                       sex, HE4, pmax, okb);
        }
        if (!okb) {
            okf = 0;
            if (box_ok && lane == 0) box_ok[box] = 0;
        }
        if (le - lb <= S) {
            double* dst = tex + (int64_t)it * HE4;
            for (int i = lane; i < NC * nh(P); i += 64) dst[4 * (i / NC) + i % NC] += W.acc[i];
        } else {
            double* dst = part + (int64_t)at * (NC * nh(P));
            for (int i = lane; i < NC * nh(P); i += 64) dst[i] = W.acc[i];
        }
        wave_sync();
    }
    if (lane == 0) {
        atomicMax(flags, pmax);
        if (!okf) atomicAnd(flags + 1, 0);
    }
}

// adds the chunks of each of the pass's boxes of more than one, in chunk order, to its target's expansion, and sets the
// counter back for the next pass
template <int CAP, bool LH>
__global__ __launch_bounds__(256) void k_m2l_mx_sum(const int32_t* __restrict__ m2l_targets,
                                                    const int64_t* __restrict__ m2l_offsets, double* __restrict__ tex,
                                                    const double* __restrict__ part, int w0, int w1, int P, int PE,
                                                    int32_t* __restrict__ flags) {
    constexpr int S = m2l_chunk(CAP, LH), NC = LH ? 4 : 2;
    const int box = blockIdx.x;
    if (box == 0 && threadIdx.x == 0) flags[2] = 0;
    const int64_t l0 = m2l_offsets[box], l1 = m2l_offsets[box + 1], first = mx_first_slot(l0, box, S);
    if (l1 - l0 <= S || first < w0 || first >= w1) return;
    const int64_t n = (l1 - l0 + S - 1) / S;
    const int len = NC * nh(P);
    const double* src = part + (first - w0) * len;
    double* dst = tex + (int64_t)m2l_targets[box] * (4 * (int64_t)nh(PE));
    for (int i = threadIdx.x; i < len; i += 256) {
        double v = src[i];
        for (int64_t c = 1; c < n; ++c) v += src[c * len + i];
        dst[4 * (i / NC) + i % NC] += v;
    }
}

template <int CAP, bool LH, int NW, bool ERR>
static void launch_m2l_mx(Context& C, int p, int pe, const Lists& Ls, const Tree& st, Tree& tt_dst, const ErrParams& E,
                          const int32_t* perm, int32_t* flags, const TablePtrs& tb) {
    auto kfn = k_m2l_mx<CAP, LH, NW, ERR>;
    const size_t sh = mx_lds_bytes<CAP, LH>(NW);
    HIP_CHECK(hipFuncSetAttribute((const void*)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sh));
    int per_cu = 0;
    HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kfn), 64 * NW, sh));
    if (!C.n_cu) HIP_CHECK(hipDeviceGetAttribute(&C.n_cu, hipDeviceAttributeMultiprocessorCount, C.device));
    constexpr int S = m2l_chunk(CAP, LH);
    // one slot past the last box's first for each of its chunks (its list may end inside a chunk)
    const int64_t slots = mx_first_slot(Ls.n_m2l, Ls.n_m2l_targets, S), len = (LH ? 4 : 2) * nh(p);
    const int64_t span = (st.n_branches + S - 1) / S;
    const int64_t room = std::max<int64_t>(M2L_PART_BYTES / (int64_t)(len * sizeof(double)), 2 * span);
    const int64_t pass = slots <= room ? slots : room - span, held = std::min(slots, room);
    C.m2l_part.resize((size_t)(held * len));
    const int64_t want = (held + NW - 1) / NW;
    const unsigned grid = (unsigned)std::max<int64_t>(1, std::min<int64_t>(want, (int64_t)std::max(per_cu, 1) * C.n_cu));
    // The counter is one address for all 8 XCDs and takes an increment about every 14 ns. Up to cap 12 a slot is less work
    // than that over 2048-3072 wavefronts (4M Plummer sphere, order 8: 18.3 ms with one increment per slot, 9.0 ms with
    // several), so a wavefront takes two to sixteen at a time, a sixth of its share; above, a slot is ten times as long
    // (1M ring, order cap 20: 20.3 ms with one, 21.8 ms with several). With a wavefront for every slot there is no counter
    // (grab 0): a small launch otherwise spends a third of its time on it.
    const int64_t waves = (int64_t)grid * NW, share = held / waves;
    const int grab = held <= waves ? 0 : CAP <= 12 && share >= 4 ? (int)std::max<int64_t>(2, std::min<int64_t>(16, share / 6)) : 1;
    for (int64_t w0 = 0; w0 < slots; w0 += pass) {
        const int64_t w1 = std::min(slots, w0 + pass);
        kfn<<<grid, 64 * NW, sh, C.stream>>>(Ls.m2l_targets.data(), Ls.m2l_offsets.data(), Ls.m2l_s.data(), tt_dst.branches.data(),
                                             st.branches.data(), st.expansions.data(), tt_dst.expansions.data(), C.m2l_part.data(),
                                             (int)Ls.n_m2l_targets, (int)w0, (int)w1, (int)std::min(slots, w1 + span), grab, p, pe,
                                             E, perm, Ls.m2l_order.data(), flags,
                                             Ls.track_box_ok ? const_cast<int32_t*>(Ls.m2l_box_ok.data()) : nullptr, tb);
        LAUNCH_CHECK();
        k_m2l_mx_sum<CAP, LH><<<(unsigned)Ls.n_m2l_targets, 256, 0, C.stream>>>(
            Ls.m2l_targets.data(), Ls.m2l_offsets.data(), tt_dst.expansions.data(), C.m2l_part.data(), (int)w0, (int)w1, p, pe, flags);
        LAUNCH_CHECK();
    }
}


static constexpr int MX_NW = 4;   // wavefronts per workgroup

// the launch at order p <= CAP (CAP the smallest instantiated cap >= p). Fixed orders and error-controlled ones have an
// engine each, so that the first holds none of the tests' values (order cap 8: 4,075 instructions and 166 registers
// against 6,595 and 208 with the tests). Degree loops of fixed length (order equal to the cap) were dropped: without
// the branch between degrees the scheduler mixes them and spills.
template <int CAP>
void run_m2l_mx_cap(Context& C, int p, bool LH, const Lists& Ls, const Tree& st, Tree& tt_dst, const ErrParams& E,
                    const int32_t* perm, int32_t* flags, const TablePtrs& tb) {
    auto run = [&](auto lh) {
        constexpr bool L = decltype(lh)::value;
        if (E.kind != 0) launch_m2l_mx<CAP, L, MX_NW, true>(C, p, p, Ls, st, tt_dst, E, perm, flags, tb);
        else launch_m2l_mx<CAP, L, MX_NW, false>(C, p, p, Ls, st, tt_dst, E, perm, flags, tb);
    };
    if (LH) run(std::true_type());
    else run(std::false_type());
}

}  // namespace fmmhip
