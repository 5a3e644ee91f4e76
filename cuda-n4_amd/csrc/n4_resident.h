// n4_resident.h -- the whole level/iteration loop of a correction in one
// launch (included by n4_kernels.hip; the host emulation build takes the LDS
// layout and the factor tables only).
//
// One workgroup of 1024 threads per compute unit.  A volume is worked on by
// a team of workgroups that stay on it from its first iteration to its last
// and meet at three team barriers per iteration (range of logU known;
// histogram complete; fit numerator complete), in place of five launches.
//
// What bounds it: the chain of one iteration -- three barriers (2.2 us each),
// the FP64 Wiener step (7.6 us), and per phase one round trip to L2 -- and, for large volumes,
// the vector work per foreground voxel.  So
//  * only the foreground is worked on: a strip (the row tile of a slab that
//    the step kernels give one workgroup) is cut into units of 16 rows, each
//    by the z range that holds its foreground, and logU lives in a packed
//    copy of the units (tiles of 16 rows x 16 z, four voxels per lane), so
//    every access is one aligned 16-byte load per lane;
//  * that lane layout is the operand layout of the matrix instructions of
//    both contractions (fit: A operand, a row of voxels per row; evaluation:
//    result, a row of voxels per column), so voxels go from memory to the
//    matrix cores and back without a pass through LDS;
//  * the factor tables of a level stay in LDS for all its iterations;
//  * every workgroup runs the Wiener step and forms the lattice increment
//    it needs itself, which costs less than the barrier it saves.
//
// Same bits as the step kernels: the FP32 matrix instruction
// (v_mfma_f32_16x16x4_f32) accumulates its four products as a chain of FMAs
// in k order, so with k ascending along the contracted axis it repeats the
// scalar loops of body_fit and eval_chunks, and terms left out (voxels
// outside a unit, zero factors) are exact zeros; the BF16 forms issue
// fit_mfma_tile's instructions on the same blocks of 32 z and 16 rows in the
// same order.  Only the FP64 convergence sums have another order.
//
// Voxel order in a tile (lane = 16 g4 + r16, element j):
//   FP32: row y0 + 4 (r16 & 3) + r16 / 4, z = zlo + 16 t + 4 j + g4
//   BF16: row y0 + r16, z = zlo + 16 t + 4 g4 + j: quad 16 a + r16 of a unit
//   holds z = zlo + 4 a .., so the fit reads the 8 z of a lane's operand on
//   blocks of 32 z from z = 0 as two quads, whatever zlo
//
// Chunks: a volume's strips are split into `nchunk` runs of about equal tile
// counts, one per workgroup of a full team.  Floating-point sums that cross
// units are formed per strip or per chunk in a fixed order and combined as
// integers or in chunk order, so the results do not depend on how many
// workgroups the team got.
//
// No workgroup waits for one that may not run: a team is formed by the
// workgroups that arrive (tickets in volume order), and the wait for the
// rest of the team is bounded (kResJoinTicks), after which it runs with the
// members it has.  Every other wait is bounded as well (kSpinLimit).
#pragma once

namespace n4 {

constexpr int kResThreads = kResBlock;
constexpr int kResWaves = kResThreads / 64;
constexpr int kResBr = 20;  // row stride of a wave's y-contracted block (16-byte rows, distinct banks)
constexpr uint32_t kResClosed = 0x80000000u;
// 100 MHz clock: 1 ms, the time that other streams' kernels take to leave the
// compute units (with 200 us the slowest call of four callers side by side,
// batch64, two head256 and a 64^3 volume, took 30 ms in place of 12).
constexpr uint64_t kResJoinTicks = 100000;

#define N4_PHASE __device__ __attribute__((noinline))
#define N4_PHASE_HD __host__ __device__ __attribute__((noinline))

// One unit of the current batch in LDS, with its slab's x factors.
struct alignas(16) ResLUnit {
    int32_t x, y0, zlo, tile;
    int32_t nt;
    int32_t cls;  // BF16: the wave of fit_mfma_tile that sums this unit, (row group of the strip) % 4
    int32_t b;    // first control plane of slab x
    int32_t pad;
    float w[4];   // evaluation factors
    float f[4];   // fit factors (w^3/sum w^2, or w^2 while the denominator is formed)
};

// What the phases of a volume read, in LDS: offsets of the LDS arrays,
// global buffers, the workgroup's share and the current level.  All values
// are the same for every lane.
struct alignas(16) ResCtx {
    // LDS arrays (byte offsets)
    uint32_t E;     // [nbins] E table (FP32)
    uint32_t Ed;    // [nbins + 1][2] E[i], E[i + 1] - E[i]; from the last bin on E, 0
    uint32_t acc;   // [lmax] fixed-point numerator of the workgroup's planes (zero between fits)
    uint32_t lres;  // [lmax] increment planes of the workgroup's slabs
    // evaluation factors.  y: row = position, 16 control points in the order
    // 4 * (c & 3) + (c >> 2), so that a lane's four operands are one 16-byte
    // read; z: the position's four factors in the order 1, 0, 2, 3, and its
    // first control point
    uint32_t wy, zw, zb;
    // fit factors of 16 control points.  FP32: [c][pos % 4][pos / 4], rows of
    // pzs / pys (odd: the 64 lanes' reads fall in different banks); BF16 hi
    // and lo halves: [c][pos], rows of pzs / pys halves
    uint32_t pz, pzl, py, pyl;
    uint32_t cb;    // [nchunk + 1][2] first unit and first tile of the own chunks
    uint32_t lu;    // [nbatch] ResLUnit
    uint32_t sf;    // [nbatch + 2] strips of the batch, then each strip's first unit and the end
    uint32_t tick;  // phase clocks of the leader
    uint32_t red;   // [4 * kResWaves] doubles
    // union: set-up arrays | histogram copies | FFT | T1 slots (1 KB per unit
    // of a batch) | evaluation: a block of 16 x kResBr floats per wave
    uint32_t u, ubytes;
    int32_t hc;     // histogram copies
    int32_t pzs, pys;
    // global buffers
    float* xq;
    const uint8_t* mq;
    const float* cq;
    const ResUnit* ulist;
    uint64_t* numfx;
    uint64_t* hist;
    double* den;
    double* lat;  // the level's lattice
    double* cpart;
    const D2* twiddle;
    double fwhm, noise;
    const AxisEntry* ax[3];
    // plan and share
    int32_t Y, Z, nbatch, wtile_rows, wtiles_x, num_copies, lmax, hist_copies;
    int32_t nb, P, offset, nch, rank, m;
    int32_t c0, c1;       // own chunks
    int32_t U0, U1;       // their units
    int32_t T0, T1;       // and tiles
    int32_t single;       // one chunk, whose units fit one batch: the list stays in LDS for a whole level
    int32_t x0, x1;       // first and last own slab
    // level
    int32_t Cy, Cz, L;
    int32_t pa, np;       // control planes of the own slabs
    int32_t o0, o1;       // control points whose update this workgroup owns
};

typedef const N4_LDS ResCtx* CtxP;
typedef N4_LDS unsigned char* LdsP;

HD uint32_t uni(uint32_t v) {
#ifdef N4_DEVICE_PASS
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
#else
    return v;
#endif
}
HD int uni(int v) { return (int)uni((uint32_t)v); }
template <class T>
HD T* uni(T* p) {
    const uint64_t v = (uint64_t)p;
    return (T*)((uint64_t)uni((uint32_t)v) | ((uint64_t)uni((uint32_t)(v >> 32)) << 32));
}
// LDS base and context of a phase function (its arguments arrive in vector
// registers).
HD LdsP res_base(LdsP smem) {
#ifdef N4_DEVICE_PASS
    return (LdsP)(uintptr_t)uni((uint32_t)(uintptr_t)smem);
#else
    return smem;
#endif
}
HD CtxP res_ctx(LdsP base) { return reinterpret_cast<CtxP>(base + kResBcBytes); }
template <class T>
HD N4_LDS T* lds_at(LdsP base, uint32_t off) {
    return reinterpret_cast<N4_LDS T*>(base + uni(off));
}

// LDS layout: offsets into o (nullable), size returned.
HD size_t carve_res(const VolDesc& V, int nbins, int P, int prec, ResCtx* o) {
    const int Y = V.W[1], Z = V.W[2];
    const int L = V.lev[V.nlevels - 1].L;
    size_t off = kResBcBytes + sizeof(ResCtx);
    auto take = [&](size_t bytes) {
        off = align16(off);
        const size_t r = off;
        off += bytes;
        return (uint32_t)r;
    };
    ResCtx c;
    c.red = take(sizeof(double) * 4 * kResWaves);
    c.tick = take(sizeof(uint64_t) * kPhases);
    c.E = take(sizeof(float) * nbins);
    c.Ed = take(sizeof(float) * 2 * (nbins + 1));
    c.acc = take(sizeof(uint64_t) * L);
    c.lres = take(sizeof(float) * L);
    c.zw = take(sizeof(float) * 4 * (Z + 16));
    c.zb = take(sizeof(int) * (Z + 16));
    c.wy = take(sizeof(float) * 16 * (Y + 16));
    if (prec == 0) {
        c.pzs = (((Z + 16 + 3) >> 2) + 4) | 1;
        c.pys = (((Y + 16 + 3) >> 2) + 4) | 1;
        c.pz = take(sizeof(float) * 64 * c.pzs);
        c.py = take(sizeof(float) * 64 * c.pys);
        c.pzl = c.pyl = 0;
    } else {
        c.pzs = round_up(Z, 32) + 8;
        c.pys = round_up(Y, 16) + 4;
        c.pz = take(sizeof(unsigned short) * 16 * c.pzs);
        c.pzl = take(sizeof(unsigned short) * 16 * c.pzs);
        c.py = take(sizeof(unsigned short) * 16 * c.pys);
        c.pyl = take(sizeof(unsigned short) * 16 * c.pys);
    }
    c.cb = take(sizeof(int) * 2 * (V.res.nchunk + 1));
    c.lu = take(sizeof(ResLUnit) * V.res.nbatch);
    c.sf = take(sizeof(int) * (V.res.nbatch + 2));
    size_t um = (size_t)V.res.nbatch * 1024;
    const size_t fft = wiener_lds(P);
    const size_t setup = (size_t)2 * (V.W[0] + 1) * sizeof(int) + (size_t)2 * Y * sizeof(int) + 64;
    const size_t br = (size_t)kResWaves * 16 * kResBr * sizeof(float);
    um = um > fft ? um : fft;
    um = um > setup ? um : setup;
    um = um > br ? um : br;
    // as many histogram copies as the union holds anyway, 8 at least
    const size_t hone = sizeof(unsigned long long) * (size_t)(nbins + 1);
    um = um > 8 * hone ? um : 8 * hone;
    c.hc = um >= 32 * hone ? 32 : (um >= 16 * hone ? 16 : 8);
    c.u = take(um);
    c.ubytes = (uint32_t)um;
    if (o) *o = c;
    return align16(off);
}

// Factor tables of a level (kf 2: w^2 for the denominator, 1: w^3/sum w^2
// and the evaluation factors): one position per thread, zeros outside the
// position's 4-point support and past the grid.
template <int PREC>
N4_PHASE_HD void res_tables(LdsP smem, int kf) {
    const LdsP base = res_base(smem);
    const CtxP C = res_ctx(base);
    const int Y = uni(C->Y), Z = uni(C->Z), pzs = uni(C->pzs), pys = uni(C->pys);
    const AxisEntry* axz = uni(C->ax[2]);
    const AxisEntry* axy = uni(C->ax[1]);
    N4_LDS float* zw = lds_at<float>(base, C->zw);
    N4_LDS int* zb = lds_at<int>(base, C->zb);
    N4_LDS float* wy = lds_at<float>(base, C->wy);
    // positions the tables hold (past the grid: zeros): the evaluation's go 16
    // past the grid, where a unit's last tile or block of rows may reach, the
    // fit's to the end of their rows
    const int fz = PREC == 0 ? 4 * pzs : pzs, fy = PREC == 0 ? 4 * pys : pys;
    const int npz = fz > Z + 16 ? fz : Z + 16, npy = fy > Y + 16 ? fy : Y + 16;
    BLOCK_FOR_N(t, kResThreads)
    for (int e = t; e < npz + npy; e += kResThreads) {
        const bool isz = e < npz;
        const int pos = isz ? e : e - npz;
        const int n = isz ? Z : Y;
        const int st = isz ? pzs : pys;
        const uint32_t tab = isz ? C->pz : C->py, tabl = isz ? C->pzl : C->pyl;
        const AxisEntry* ax = isz ? axz : axy;
        float f[4] = {0.0f, 0.0f, 0.0f, 0.0f}, w[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        int b = 0;
        if (pos < n) {
            const AxisEntry& a = ax[pos];
            b = a.b;
            UNROLL for (int k = 0; k < 4; ++k) {
                f[k] = kf == 2 ? a.q[k] : a.p[k];
                w[k] = a.w[k];
            }
        }
        const bool ev = kf != 2 && pos < n + 16, fit = pos < (isz ? fz : fy);
        if (ev && isz) {
            // the factors of row z in the association of eval_chunks (see res_eval);
            // past the grid zeros, in the last span
            UNROLL for (int k = 0; k < 4; ++k) zw[4 * pos + k] = w[k < 2 ? 1 - k : k];
            zb[pos] = pos < n ? b : axz[n - 1].b;
        }
        for (int c = 0; c < 16; ++c) {
            const int k = c - b;
            float fv = 0.0f, wv = 0.0f;
            UNROLL for (int a = 0; a < 4; ++a)
                if (k == a) {
                    fv = f[a];
                    wv = w[a];
                }
            if (!fit) {
            } else if constexpr (PREC == 0) {
                lds_at<float>(base, 0)[tab / 4 + (4 * c + (pos & 3)) * st + (pos >> 2)] = fv;
            } else {
                unsigned short h, l;
                bf16_split(fv, h, l);
                lds_at<unsigned short>(base, 0)[tab / 2 + c * st + pos] = h;
                lds_at<unsigned short>(base, 0)[tabl / 2 + c * st + pos] = l;
            }
            if (ev && !isz) wy[pos * 16 + 4 * (c & 3) + (c >> 2)] = wv;
        }
    }
    BLOCK_END
}

}  // namespace n4

#ifndef N4_EMULATE
namespace n4 {

__device__ inline f32x4 mma_f32(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Phase clocks of a team's leader (device clock), kept in LDS by thread 0.
struct ResTimer {
    N4_LDS unsigned long long* slots;
    bool on;
    uint64_t last;
    __device__ void mark(int phase) {
        if (!on || threadIdx.x != 0) return;
        const uint64_t now = PhaseTimer::now();
        slots[phase] += now - last;
        last = now;
    }
};

// What the Wiener step needs besides the histogram -- the Gaussian and the
// twiddles -- laid into its buffers by the waves that have nothing to do
// while the first polls the barrier of the complete histogram (Wiener step
// 8.25 -> 7.6 us).
template <int P>
__device__ inline void res_wiener_ready_p(LdsP u, const RunParams& rp, double slope) {
    constexpr bool PAD = fft_pad(P);
    const WienerLds L = carve_wiener<P, PAD>(u);
    const WienerGauss G = wiener_gauss(rp, slope);
    for (int j = (int)threadIdx.x - 64; j < P; j += kResThreads - 64) {
        L.tw[fft_at<PAD>(j)] = rp.twiddle[j];
        L.z[fft_at<PAD>(j)].y = wiener_gauss_at<P>(G, j);
    }
}
__device__ inline void res_wiener_ready(LdsP base, double slope) {
    const CtxP C = res_ctx(base);
    RunParams rp;
    rp.fwhm = C->fwhm;
    rp.twiddle = uni(C->twiddle);
    const LdsP u = lds_at<unsigned char>(base, C->u);
    switch (uni(C->P)) {
        case 4: res_wiener_ready_p<4>(u, rp, slope); break;
        case 8: res_wiener_ready_p<8>(u, rp, slope); break;
        case 16: res_wiener_ready_p<16>(u, rp, slope); break;
        case 32: res_wiener_ready_p<32>(u, rp, slope); break;
        case 64: res_wiener_ready_p<64>(u, rp, slope); break;
        case 128: res_wiener_ready_p<128>(u, rp, slope); break;
        case 256: res_wiener_ready_p<256>(u, rp, slope); break;
        case 512: res_wiener_ready_p<512>(u, rp, slope); break;
        default: res_wiener_ready_p<1024>(u, rp, slope); break;
    }
}


// Team barrier number gen + 1 (see team_barrier): bounded, false once the
// team has given up.
template <bool WIENER>
N4_PHASE bool res_barrier_t(uint32_t* team_, int m_, uint32_t gen, LdsP smem, double slope) {
    uint32_t* team = uni(team_);
    const int m = uni(m_);
    const LdsP base = res_base(smem);
    N4_LDS int* bc = reinterpret_cast<N4_LDS int*>(base);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    int ok = 1;
    if (m > 1 && threadIdx.x == 0)
        __hip_atomic_fetch_add(team + kRwBarrier, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (WIENER && threadIdx.x >= 64) res_wiener_ready(base, slope);
    if (m > 1 && threadIdx.x == 0) {
        const uint32_t target = (gen + 1u) * (uint32_t)m;
        for (uint32_t spins = 1; ld_agent(team + kRwBarrier) < target; ++spins) {
            __builtin_amdgcn_s_sleep(1);
            if ((spins & 63u) == 0 && (spins > kSpinLimit || ld_agent(team + kRwAbort) != 0)) {
                ok = 0;
                break;
            }
        }
        if (!ok) st_agent(team + kRwAbort, 1u);
        bc[0] = ok;
    }
    if (m == 1 && !WIENER) return true;
    __syncthreads();
    return m == 1 || uni(bc[0]) != 0;
}
__device__ inline bool res_barrier(uint32_t* team, int m, uint32_t gen, LdsP smem) {
    return res_barrier_t<false>(team, m, gen, smem, 0.0);
}

// Joins a team of n workgroups: rank (>= 0; the team's size in broadcast
// word 2); -1: the team was closed before this workgroup came; -2: gave up.
N4_PHASE int res_join(uint32_t* team, int n, LdsP smem) {
    N4_LDS int* bc = reinterpret_cast<N4_LDS int*>(res_base(smem));
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t old = __hip_atomic_fetch_add(team + kRwJoin, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        int r = (int)old;
        uint32_t size = 0;
        if (old & kResClosed) {
            r = -1;
        } else {
            const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
            bool close = old + 1u == (uint32_t)n;
            for (uint32_t spins = 0;; ++spins) {
                if (close) {
                    const uint32_t prev =
                        __hip_atomic_fetch_or(team + kRwJoin, kResClosed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (!(prev & kResClosed)) st_agent(team + kRwSize, prev);
                    close = false;
                }
                size = ld_agent(team + kRwSize);
                if (size != 0) break;
                if (spins > kSpinLimit) {
                    st_agent(team + kRwAbort, 1u);
                    r = -2;
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
                if ((spins & 15u) == 15u) close = __builtin_amdgcn_s_memrealtime() - t0 > kResJoinTicks;
            }
        }
        bc[1] = r;
        bc[2] = (int)size;
    }
    __syncthreads();
    return uni(bc[1]);
}

// Units [ub, ub + n) of the volume's list (whole strips, n <= 64) into LDS,
// with the x factors of the level (kf as above).
N4_PHASE void res_load_batch(LdsP smem, int ub, int n, int kf) {
    const LdsP base = res_base(smem);
    const CtxP C = res_ctx(base);
    const int t = (int)threadIdx.x;
    const ResUnit* ulist = uni(C->ulist);
    N4_LDS ResLUnit* lu = lds_at<ResLUnit>(base, C->lu);
    N4_LDS int* sf = lds_at<int>(base, C->sf);
    const int rows = uni(C->wtile_rows);
    if (t >= 64) return;
    const ResUnit u = ulist[ub + (t < n ? t : 0)];
    if (t < n) {
        const AxisEntry a = uni(C->ax[0])[u.x];
        ResLUnit o;
        o.x = u.x;
        o.y0 = u.y0;
        o.zlo = u.zlo;
        o.tile = u.tile;
        o.nt = u.nt;
        o.cls = (u.y0 % rows) / 16 & 3;
        o.b = a.b;
        o.pad = 0;
        for (int k = 0; k < 4; ++k) {
            o.w[k] = a.w[k];
            o.f[k] = kf == 2 ? a.q[k] : a.p[k];
        }
        lu[t] = o;
    }
    const int strip = u.x * uni(C->wtiles_x) + u.y0 / rows;
    const int prev = __shfl_up(strip, 1);
    const bool first = t < n && (t == 0 || prev != strip);
    const unsigned long long m = __ballot(first);
    if (first) sf[1 + __popcll(m & ((1ull << t) - 1ull))] = t;
    if (t == 0) {
        sf[0] = __popcll(m);
        sf[1 + __popcll(m)] = n;
    }
}

// Units from ub that one batch takes, of those before u1: as many whole
// strips as fit (the next batch starts at ub + the result).
__device__ inline int res_batch_len(CtxP C, int ub, int u1) {
    const int nb = uni(C->nbatch), rows = uni(C->wtile_rows);
    if (u1 - ub <= nb) return u1 - ub;
    // the last unit of the window that starts a strip
    const ResUnit* ulist = uni(C->ulist);
    const int lane = (int)threadIdx.x & 63;
    const int i = lane < nb ? lane : nb - 1;
    const ResUnit u = ulist[ub + i + 1], p = ulist[ub + i];
    const bool first = u.x != p.x || u.y0 / rows != p.y0 / rows;
    const unsigned long long m = __ballot(first && lane < nb);
    return uni(64 - __clzll(m));
}

// fit_input of one voxel with the paired E table (same operations: the
// difference of neighbouring entries is formed once per bin, and from the
// last bin on the entry itself comes back as fma(0, ., E)).  on: all ones
// where the voxel counts, else 0; as a bit mask it keeps the table reads of
// all voxels in flight (a select becomes a branch around each read, with a
// wait of its own; FP32, 256 x 256 x 176 at shrink 4: 2.17 against 2.19 ms).
template <bool DEN>
__device__ inline float res_input(int on, float xv, const Remap& R, const N4_LDS float* Ed) {
    if constexpr (DEN) return __int_as_float(on & __float_as_int(1.0f));
    float c = (xv - R.bmin) * R.islope;
    c = fminf(fmaxf(c, 0.0f), (float)R.nb);
    const int idx = (int)c;
    const float fr = c - (float)idx;
    typedef float f2 __attribute__((ext_vector_type(2)));
    const f2 e = *reinterpret_cast<const N4_LDS f2*>(Ed + 2 * idx);
    return __int_as_float(on & __float_as_int(xv - fmaf(e[1], fr, e[0])));
}
// Bit j of a quad's mask byte as all ones or 0.
__device__ inline int res_on(uint32_t m, int j) { return (int)(m << (31 - j)) >> 31; }

// A pair of floats as BF16, round to nearest even, low half first.
__device__ inline uint32_t res_pk(float a, float b) {
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{a, b}, bf2));
}

// T1 of one unit by one wave: the z contraction of g = fit_input over the
// unit's voxels.  Row 4 g4 + i of the result is a row of voxels in the tile
// order, column lane % 16 a control point along z.  pz: the lane's row of
// the factor table.
template <int PREC, bool DEN>
__device__ inline f32x4 res_fit_unit(const float* xq, const uint8_t* mq, const float* cq, const N4_LDS float* Ed,
                                     const N4_LDS unsigned char* pz, const N4_LDS unsigned char* pzl, int tile, int nt,
                                     int zlo, uint32_t live, const Remap& rm) {
    const int lane = (int)threadIdx.x & 63, r16 = lane & 15, g4 = lane >> 4;
    f32x4 t1 = f32x4{0, 0, 0, 0};
    if constexpr (PREC == 0) {
        const size_t q0 = (size_t)tile * 64 + lane;
        constexpr int kAhead = 4;  // tiles in flight
        for (int tb = 0; tb < nt; tb += kAhead) {
            F4 xs[kAhead], cs[kAhead];
            uint32_t ms[kAhead];
            UNROLL for (int k = 0; k < kAhead; ++k) {
                const bool ok = tb + k < nt;
                const size_t q = q0 + (size_t)(ok ? tb + k : tb) * 64;
                ms[k] = gp(mq)[q] & (ok ? live : 0u);
                xs[k] = load_quad(xq + 4 * q);
                if (cq) cs[k] = load_quad(cq + 4 * q);
            }
            const N4_LDS float* b = reinterpret_cast<const N4_LDS float*>(pz) + (zlo >> 2) + 4 * tb;
            float g[kAhead][4], f[kAhead][4];
            UNROLL for (int k = 0; k < kAhead; ++k) UNROLL for (int j = 0; j < 4; ++j) {
                g[k][j] = res_input<DEN>(res_on(ms[k], j), xs[k].v[j], rm, Ed);
                f[k][j] = b[4 * k + j];
            }
            if (cq)
                UNROLL for (int k = 0; k < kAhead; ++k) UNROLL for (int j = 0; j < 4; ++j)
                    if ((ms[k] >> j) & 1u) g[k][j] *= cs[k].v[j];
            // (tiles past the unit's end: zeros, which leave the chain as it is)
            UNROLL for (int k = 0; k < kAhead; ++k) {
                if (tb + k >= nt) break;
                UNROLL for (int j = 0; j < 4; ++j) t1 = mma_f32(g[k][j], f[k][j], t1);
            }
        }
    } else {
        // blocks of 32 z from z = 0, two in flight
        const int T0 = zlo >> 5, T1 = (zlo + 16 * nt + 31) >> 5;
        for (int T = T0; T < T1; T += 2) {
            F4 xs[4];
            uint32_t ms[4];
            UNROLL for (int k = 0; k < 4; ++k) {
                const int a = ((32 * (T + (k >> 1)) + 8 * g4 - zlo) >> 2) + (k & 1);
                const bool ok = a >= 0 && a < 4 * nt;
                const size_t q = (size_t)tile * 64 + (ok ? 16 * a : 0) + r16;
                ms[k] = gp(mq)[q] & (ok ? live : 0u);
                xs[k] = load_quad(xq + 4 * q);
            }
            // (a branch per voxel here: its waits, one quad at a time, cost
            // less than all sixteen table reads at once -- 64-volume batch
            // 6.74 against 6.93 ms)
            auto in = [&](int k, int j) {
                return (ms[k] >> j) & 1u ? res_input<DEN>(-1, xs[k].v[j], rm, Ed) : 0.0f;
            };
            UNROLL for (int k = 0; k < 4; k += 2) {
                if (T + (k >> 1) >= T1) break;
                uint32_t h4[4], l4[4];
                UNROLL for (int p = 0; p < 4; ++p) {
                    const int kk = k + (p >> 1), j = 2 * (p & 1);
                    const float g0 = in(kk, j), g1 = in(kk, j + 1);
                    const uint32_t h = res_pk(g0, g1);
                    h4[p] = h;
                    if constexpr (PREC == 2)
                        l4[p] = res_pk(g0 - __uint_as_float(h << 16), g1 - __uint_as_float(h & 0xffff0000u));
                    else
                        l4[p] = 0;
                }
                typedef uint32_t u4 __attribute__((ext_vector_type(4)));
                const u16x8 ah = __builtin_bit_cast(u16x8, u4{h4[0], h4[1], h4[2], h4[3]});
                const u16x8 al = __builtin_bit_cast(u16x8, u4{l4[0], l4[1], l4[2], l4[3]});
                const int o = 2 * (32 * (T + (k >> 1)) + 8 * g4);
                const u16x8 bh = *reinterpret_cast<const N4_LDS u16x8*>(pz + o);
                const u16x8 bl = *reinterpret_cast<const N4_LDS u16x8*>(pzl + o);
                t1 = mma_k32p<PREC, true>(ah, al, bh, bl, t1);
            }
        }
    }
    return t1;
}

// rint(v) as a 64-bit integer, read from the low bits of v + 1.5 2^52; exact
// for |v| < kResFixedMax.
constexpr double kResFixedMax = 2251799813685248.0;  // 2^51
__device__ inline unsigned long long res_fixed(double v) {
    constexpr double kMagic = 6755399441055744.0;
    return (unsigned long long)(__double_as_longlong(v + kMagic) - __double_as_longlong(kMagic));
}

// Fit of the workgroup's chunks, per batch of whole strips: T1 of every unit
// into its LDS slot; per strip one wave runs the chain T2 += Py T1 over its
// units in row order (BF16: a chain per wave of fit_mfma_tile, added in wave
// order) and adds T2, weighted by the four x factors and rounded to fixed
// point one by one (scatter_numerator), to the planes in LDS; then one
// atomic per control point into the numerator copy of the chunk.  (Summing
// the strips per control point instead, each thread walking the batch's
// strips, took two thirds of the fit on a 64-volume batch.)
template <int PREC, bool DEN>
N4_PHASE void res_fit(LdsP smem, int degenerate_, double bmin, double slope) {
    const LdsP base = res_base(smem);
    const CtxP C = res_ctx(base);
    const int t = (int)threadIdx.x, wv = uni(t >> 6), lane = t & 63, r16 = lane & 15, g4 = lane >> 4;
    const int Cy = uni(C->Cy), Cz = uni(C->Cz), CyCz = Cy * Cz;
    const bool single = uni(C->single) != 0;
    const uint32_t live = uni(degenerate_) != 0 ? 0u : 0xffu;  // (degenerate: no residual anywhere)
    const float* xq = uni(C->xq);
    const uint8_t* mq = uni(C->mq);
    const float* cq = uni(C->cq);
    const N4_LDS float* Ed = lds_at<float>(base, C->Ed);
    const N4_LDS ResLUnit* lu = lds_at<ResLUnit>(base, C->lu);
    const N4_LDS int* sf = lds_at<int>(base, C->sf);
    const N4_LDS int* cb = lds_at<int>(base, C->cb);
    N4_LDS unsigned long long* acc = lds_at<unsigned long long>(base, C->acc);
    N4_LDS float* slot = lds_at<float>(base, C->u);
    const int pzs = uni(C->pzs), pys = uni(C->pys);
    // the lane's rows of the factor tables
    const LdsP pz = lds_at<unsigned char>(base, C->pz) + (PREC == 0 ? 4 * (4 * r16 + g4) * pzs : 2 * r16 * pzs);
    const LdsP pzl = lds_at<unsigned char>(base, C->pzl) + 2 * r16 * pzs;
    const LdsP py = lds_at<unsigned char>(base, C->py) + (PREC == 0 ? 4 * (4 * r16 + g4) * pys : 2 * (r16 * pys + 4 * g4));
    const LdsP pyl = lds_at<unsigned char>(base, C->pyl) + 2 * (r16 * pys + 4 * g4);
    const Remap rm = make_remap(nullptr, bmin, slope, uni(C->nb));
    constexpr int kCls = PREC == 0 ? 1 : 4;
    const int c0 = uni(C->c0), c1 = uni(C->c1);
    for (int c = c0; c < c1; ++c) {
        const int u1 = uni(cb[2 * (c - c0) + 2]);
        for (int ub = uni(cb[2 * (c - c0)]), n; ub < u1; ub += n) {
            n = single ? u1 - ub : res_batch_len(C, ub, u1);
            if (!single) {
                __syncthreads();
                res_load_batch(smem, ub, n, DEN ? 2 : 1);
                __syncthreads();
            }
            for (int i = wv; i < n; i += kResWaves) {
                const f32x4 a = res_fit_unit<PREC, DEN>(xq, mq, cq, Ed, pz, pzl, uni(lu[i].tile), uni(lu[i].nt),
                                                        uni(lu[i].zlo), live, rm);
                *reinterpret_cast<N4_LDS f32x4*>(slot + i * 256 + 4 * lane) = a;
            }
            __syncthreads();
            const int ns = uni(sf[0]), pa = uni(lu[0].b), np = uni(lu[n - 1].b) + 4 - pa;
            for (int k = wv; k < ns; k += kResWaves) {
                const int s0 = uni(sf[1 + k]), s1 = uni(sf[2 + k]);
                f32x4 v[kCls];
                UNROLL for (int w = 0; w < kCls; ++w) v[w] = f32x4{0, 0, 0, 0};
                for (int i = s0; i < s1; ++i) {
                    const f32x4 t1 = *reinterpret_cast<const N4_LDS f32x4*>(slot + i * 256 + 4 * lane);
                    const int y0 = uni(lu[i].y0);
                    if constexpr (PREC == 0) {
                        const N4_LDS float* a = reinterpret_cast<const N4_LDS float*>(py) + (y0 >> 2);
                        UNROLL for (int j = 0; j < 4; ++j) v[0] = mma_f32(a[j], t1[j], v[0]);
                    } else {
                        i16x4 bh, bl;
                        to_op4<PREC>(t1, bh, bl);
                        const i16x4 a_h = *reinterpret_cast<const N4_LDS i16x4*>(py + 2 * y0);
                        const i16x4 a_l = *reinterpret_cast<const N4_LDS i16x4*>(pyl + 2 * y0);
                        const int cls = uni(lu[i].cls);
                        UNROLL for (int w = 0; w < kCls; ++w)
                            if (cls == w) v[w] = mma_k16p<PREC, false>(bh, bl, a_h, a_l, v[w]);
                    }
                }
                // T2[cy][cz]: rows 4 g4 + i, column r16 (BF16: the waves' sums in
                // wave order), into the strip's four planes
                const N4_LDS ResLUnit& U = lu[s0];
                N4_LDS unsigned long long* dp = acc + (uni(U.b) - pa) * CyCz + 4 * g4 * Cz + r16;
                double f[4], t2[4], big = 0.0;
                UNROLL for (int p = 0; p < 4; ++p) f[p] = (double)U.f[p];
                UNROLL for (int i = 0; i < 4; ++i) {
                    float x = v[0][i];
                    if constexpr (PREC != 0) x = ((x + v[1][i]) + v[2][i]) + v[3][i];
                    t2[i] = (double)x;
                    big = fmax(big, fabs(t2[i]));
                }
                // (the factors are at most 1; NaN counts as wide)
                const bool wide = __ballot(!(big * kNumScale < kResFixedMax)) != 0;
                UNROLL for (int i = 0; i < 4; ++i) {
                    if (4 * g4 + i >= Cy || r16 >= Cz) continue;
                    if (!wide) {
                        UNROLL for (int p = 0; p < 4; ++p)
                            lds_add_u64(dp + p * CyCz + i * Cz, res_fixed(f[p] * t2[i] * kNumScale));
                    } else {
                        for (int p = 0; p < 4; ++p)
                            lds_add_u64(dp + p * CyCz + i * Cz,
                                        (unsigned long long)(long long)rint((double)U.f[p] * t2[i] * kNumScale));
                    }
                }
            }
            __syncthreads();
            uint64_t* dst = uni(C->numfx) + (size_t)(c % uni(C->num_copies)) * uni(C->lmax) + (size_t)pa * CyCz;
            for (int e = t; e < np * CyCz; e += kResThreads) {
                const unsigned long long q = acc[e];
                acc[e] = 0ull;
                if (q != 0) global_add_u64(dst + e, q);
            }
            if (!single) __syncthreads();  // the slots and the unit list are reused
        }
    }
}

// u = exp(-d) - 1: for |d| <= 0.5 by the Taylor series through d^8 (the next
// term is below 2^-26 of the result), else through expm1f.
__device__ inline void res_expm1(f32x4 d, float (&u)[4]) {
    UNROLL for (int j = 0; j < 4; ++j) {
        const float x = -d[j];
        float q = fmaf(x, 1.0f / 40320.0f, 1.0f / 5040.0f);
        q = fmaf(x, q, 1.0f / 720.0f);
        q = fmaf(x, q, 1.0f / 120.0f);
        q = fmaf(x, q, 1.0f / 24.0f);
        q = fmaf(x, q, 1.0f / 6.0f);
        q = fmaf(x, q, 0.5f);
        u[j] = fmaf(x * x, q, x);
    }
    const float big = fmaxf(fmaxf(fabsf(d[0]), fabsf(d[1])), fmaxf(fabsf(d[2]), fabsf(d[3])));
    if (!(big <= 0.5f)) {
#pragma unroll 1
        for (int j = 0; j < 4; ++j) u[j] = expm1f(-d[j]);
    }
}

// Field increment, logU update and convergence sums of the workgroup's
// chunks (the lattice increment planes from plane pa are in S.lres); one
// partial quadruple per chunk.  Per unit the wave forms the y-contracted
// block Br[y][cz] on the matrix cores and parks it in LDS; per tile,
// d[z][y] = sum_c wz[z][c] Br[y][c] is one matrix instruction for every span
// of the tile's z range: rows z outside the span have zero factors there,
// and the four control points of a span are taken in the order 1, 0, 2, 3,
// the association the compiler gives eval_chunks' sum of products
// (fma(w0, b0, w1 b1), then the others).
template <int PREC>
N4_PHASE void res_eval(LdsP smem) {
    const LdsP base = res_base(smem);
    const CtxP C = res_ctx(base);
    const int t = (int)threadIdx.x, wv = uni(t >> 6), lane = t & 63, r16 = lane & 15, g4 = lane >> 4;
    const int Cy = uni(C->Cy), Cz = uni(C->Cz), CyCz = Cy * Cz;
    const bool single = uni(C->single) != 0;
    const int nsy = (Cy + 3) >> 2, zlast = Cz - 4;
    const int pr = 4 * (r16 & 3) + (r16 >> 2);
    const int ry = PREC == 0 ? pr : r16;  // this lane's row of voxels (operand column)
    const int rz = PREC == 0 ? pr : r16;  // and the z of its operand row
    const int kz = g4 < 2 ? 1 - g4 : g4;  // control point of a span in operand position g4
    float* xq = uni(C->xq) + 4 * lane;
    const uint8_t* mq = uni(C->mq) + lane;
    const N4_LDS ResLUnit* lu = lds_at<ResLUnit>(base, C->lu);
    const N4_LDS int* cb = lds_at<int>(base, C->cb);
    const N4_LDS float* wyl = lds_at<float>(base, C->wy) + 16 * ry + 4 * g4;
    const N4_LDS float* zwl = lds_at<float>(base, C->zw) + 4 * rz + g4;
    const N4_LDS int* zb = lds_at<int>(base, C->zb);
    const N4_LDS float* lres = lds_at<float>(base, C->lres);
    N4_LDS double* red = lds_at<double>(base, C->red);
    N4_LDS float* brs = lds_at<float>(base, C->u) + wv * 16 * kResBr + r16 * kResBr;
    const int c0 = uni(C->c0), c1 = uni(C->c1), pa = uni(C->pa);
    for (int c = c0; c < c1; ++c) {
        const int u0 = uni(cb[2 * (c - c0)]), u1 = uni(cb[2 * (c - c0) + 2]);
        double s1 = 0.0, s2 = 0.0;
        float mn = INFINITY, mx = -INFINITY;
        for (int ub = u0, n; ub < u1; ub += n) {
            n = single ? u1 - ub : res_batch_len(C, ub, u1);
            if (!single) {
                __syncthreads();
                res_load_batch(smem, ub, n, 1);
                __syncthreads();
            }
            // a contiguous share of the batch's tiles per wave, so a wave
            // forms the y-contracted block of few units
            const int b0 = uni(lu[0].tile), nb = uni(lu[n - 1].tile) + uni(lu[n - 1].nt) - b0;
            const int ta = b0 + nb * wv / kResWaves, te = b0 + nb * (wv + 1) / kResWaves;
            if (ta >= te) continue;
            // the unit that holds tile ta (at most 64 units in a batch)
            int i = __popcll(__ballot(lane < n && lu[lane < n ? lane : 0].tile <= ta)) - 1;
            for (int tau = ta; tau < te; ++i) {
                const N4_LDS ResLUnit& U = lu[i];
                const int utile = uni(U.tile), y0 = uni(U.y0), zlo = uni(U.zlo), ub0 = uni(U.b);
                const int uend = utile + uni(U.nt), tl = uend < te ? uend : te;
                // four tiles at a time: their loads, table reads, matrix chains
                // and series run side by side (a wave has few tiles, so one
                // tile's chain of waits would be exposed)
                constexpr int kAhead = 4;
                F4 xs[kAhead];
                uint32_t ms[kAhead];
                auto load = [&](int tau0) {
                    UNROLL for (int k = 0; k < kAhead; ++k) {
                        const bool ok = tau0 + k < tl;
                        const size_t q = (size_t)(ok ? tau0 + k : tau0) * 64;
                        ms[k] = ok ? gp(mq)[q] : 0u;
                        xs[k] = load_quad(xq + 4 * q);
                    }
                };
                load(tau);
                {
                    const N4_LDS float* lr = lres + (ub0 - pa) * CyCz + r16;
                    const f32x4 wy = *reinterpret_cast<const N4_LDS f32x4*>(wyl + 16 * y0);
                    const float w[4] = {U.w[0], U.w[1], U.w[2], U.w[3]};
                    f32x4 br = f32x4{0, 0, 0, 0};
                    UNROLL for (int s = 0; s < 4; ++s) {
                        if (s >= nsy) break;
                        const bool on = 4 * s + g4 < Cy && r16 < Cz;
                        const N4_LDS float* p = lr + (on ? (4 * s + g4) * Cz : -r16);
                        float a = 0.0f;
                        UNROLL for (int k = 0; k < 4; ++k) a += w[k] * p[k * CyCz];
                        br = mma_f32(on ? a : 0.0f, wy[s], br);
                    }
                    // rows cz = 4 g4 + i of column y: [y][cz]
                    *reinterpret_cast<N4_LDS f32x4*>(brs + 4 * g4) = br;
                }
                for (; tau < tl; tau += kAhead) {
                    float wz[kAhead];
                    int bz[kAhead], bl[kAhead], ns = 0;
                    UNROLL for (int k = 0; k < kAhead; ++k) {
                        const int z0 = zlo + 16 * ((tau + k < tl ? tau + k : tau) - utile);
                        wz[k] = zwl[4 * z0];
                        bz[k] = zb[z0 + rz];
                        bl[k] = uni(zb[z0]);
                        const int sp = uni(zb[z0 + 15]) - bl[k] + 1;
                        ns = sp > ns ? sp : ns;
                    }
                    f32x4 d[kAhead];
                    UNROLL for (int k = 0; k < kAhead; ++k) d[k] = f32x4{0, 0, 0, 0};
                    for (int s = 0; s < ns; ++s)
                        UNROLL for (int k = 0; k < kAhead; ++k) {
                            const int b = bl[k] + s < zlast ? bl[k] + s : zlast;  // (past a tile's spans: zero factors)
                            d[k] = mma_f32(bz[k] == bl[k] + s ? wz[k] : 0.0f, brs[b + kz], d[k]);
                        }
                    UNROLL for (int k = 0; k < kAhead; ++k) {
                        if (__ballot(ms[k] != 0) == 0) continue;
                        F4 o = xs[k];
                        float u[4];
                        res_expm1(d[k], u);
                        UNROLL for (int j = 0; j < 4; ++j) {
                            const bool m = (ms[k] >> j) & 1u;
                            const float lg = xs[k].v[j] - d[k][j];
                            o.v[j] = m ? lg : xs[k].v[j];
                            const double uu = (double)(m ? u[j] : 0.0f);
                            s1 += uu;
                            s2 += uu * uu;
                            mn = fminf(mn, m ? lg : INFINITY);
                            mx = fmaxf(mx, m ? lg : -INFINITY);
                        }
                        store_quad(xq + 256 * (size_t)(tau + k), o);
                    }
                    if (tau + kAhead < tl) load(tau + kAhead);
                }
                tau = tl;
            }
        }
        // the chunk's sums: wave butterflies, then the waves in order
        double v[4] = {s1, s2, (double)mn, (double)mx};
        const int ops[4] = {0, 0, 1, 2};
        UNROLL for (int sh = 32; sh > 0; sh >>= 1)
            UNROLL for (int k = 0; k < 4; ++k) v[k] = red_apply(ops[k], v[k], __shfl_xor(v[k], sh));
        if (lane == 0) UNROLL for (int k = 0; k < 4; ++k) red[4 * wv + k] = v[k];
        __syncthreads();
        if (t < 4) {
            double r = red[t];
            for (int w = 1; w < kResWaves; ++w) r = red_apply(t < 2 ? 0 : t - 1, r, red[4 * w + t]);
            st_agent(uni(C->cpart) + 4 * (size_t)c + t, r);
        }
        if (c + 1 < c1) __syncthreads();
    }
}

// Histogram of tiles [T0, T1) of the packed copy, N4.py:19-29 (as
// hist_voxel: the same bin index and share), into a global copy of the bins.
// A voxel is one LDS atomic: its count in the high 16 bits of a bin's slot,
// the share q of the next bin in the low 48 (the bin holds
// count 2^32 - sum q + sum q of the bin before).  The slots are laid out
// [bin][copy] with a lane's copy its index modulo the copies, so lanes of
// different copies fall in different LDS banks whatever their bins; with the
// two atomics per voxel and the eight bin-major copies of the step kernels
// this phase was bound by the LDS atomics (17.6 us of a 64-volume batch's
// 75 us step).  A pass takes at most kResHistTiles tiles, so that a copy's
// count stays below 2^16 even if every voxel falls in one bin.
constexpr int kResHistTiles = 2000;  // 2000 tiles x 256 voxels / 8 copies = 64000
N4_PHASE void res_hist(LdsP smem, double mn, double slope) {
    const LdsP base = res_base(smem);
    const CtxP C = res_ctx(base);
    const int t = (int)threadIdx.x, hc = uni(C->hc), nb = uni(C->nb), T0 = uni(C->T0), T1 = uni(C->T1);
    const float* xq = uni(C->xq);
    const uint8_t* mq = uni(C->mq);
    N4_LDS unsigned long long* h = lds_at<unsigned long long>(base, C->u);
    uint64_t* dst = uni(C->hist) + (size_t)(uni(C->rank) % uni(C->hist_copies)) * nb;
    const Bins B = make_bins(mn, slope, nb);
    for (int Ta = T0; Ta < T1; Ta += kResHistTiles) {
        const int Te = T1 - Ta > kResHistTiles ? Ta + kResHistTiles : T1;
        typedef unsigned long long u2 __attribute__((ext_vector_type(2)));
        for (int i = t; i < nb * hc / 2; i += kResThreads) reinterpret_cast<N4_LDS u2*>(h)[i] = u2{0ull, 0ull};
        __syncthreads();
        N4_LDS unsigned long long* hl = h + (t & (hc - 1));
        const int hs = uni(__ffs(hc) - 1);
        constexpr int kAhead = 4;
        for (int q0 = Ta * 64; q0 < Te * 64; q0 += kAhead * kResThreads) {
            F4 xs[kAhead];
            uint32_t ms[kAhead];
            UNROLL for (int k = 0; k < kAhead; ++k) {
                const int q = q0 + k * kResThreads + t;
                const bool ok = q < Te * 64;
                ms[k] = ok ? gp(mq)[q] : 0u;
                xs[k] = load_quad(xq + 4 * (size_t)(ok ? q : Ta * 64));
            }
            UNROLL for (int k = 0; k < kAhead; ++k) {
                if (__ballot(ms[k] != 0) == 0) continue;
                UNROLL for (int j = 0; j < 4; ++j) {
                    const BinShare b = bin_share(B, xs[k].v[j]);
                    if (b.in && ((ms[k] >> j) & 1u)) lds_add_u64(hl + (b.idx << hs), (1ull << 48) + b.q);
                }
            }
        }
        __syncthreads();
        // four threads per bin sum its copies; the share of the bin before comes
        // through LDS (the slot of copy 0, read by then)
        for (int i0 = 0; i0 < nb; i0 += kResThreads / 4) {
            const int i = i0 + (t >> 2), part = t & 3, per = hc >> 2;
            unsigned long long cnt = 0, sq = 0;
            if (i < nb)
                for (int k = 0; k < per; ++k) {  // (rotated by the bin: bins are a multiple of the banks apart)
                    const unsigned long long v = h[(size_t)i * hc + part * per + ((k + i) & (per - 1))];
                    cnt += v >> 48;
                    sq += v & ((1ull << 48) - 1);
                }
            UNROLL for (int sh = 1; sh < 4; sh <<= 1) {
                cnt += __shfl_xor(cnt, sh);
                sq += __shfl_xor(sq, sh);
            }
            __syncthreads();
            if (i < nb && part == 0) h[(size_t)i * hc] = sq;
            __syncthreads();
            if (i < nb && part == 0) {
                const unsigned long long s = (cnt << 32) - sq + (i > 0 ? h[(size_t)(i - 1) * hc] : 0ull);
                if (s) global_add_u64(dst + i, s);
            }
        }
        if (Te < T1) __syncthreads();
    }
}

// Cuts of the chunks at strip boundaries that keep the largest chunk small,
// where chunks hold few strips: cutting at equal tile counts leaves a chunk
// up to a strip too large, and every phase waits for it (256 x 256 x 160
// working voxels, 256 chunks of 3.6 strips: 119 tiles at most where 85 is
// the mean, 100 the least possible).  Each wave fills chunks up to a limit
// of its own, the smallest limit that suffices wins; the same in every
// member.  Chunks of many strips are even as they are, and small ones gain
// less than this costs (30 us), so they keep the equal counts (false).
// After the scan of the slabs (pt, pu in the union).
N4_PHASE bool res_even_cuts(const VolDesc* Vp, LdsP smem) {
    const VolDesc& V = *uni(Vp);
    const LdsP base = res_base(smem);
    const CtxP C = res_ctx(base);
    const int t = (int)threadIdx.x, wv = uni(t >> 6), lane = t & 63;
    const int W0 = V.W[0], nch = V.res.nchunk, c0 = uni(C->c0), c1 = uni(C->c1), rows = V.wtile_rows;
    N4_LDS int* pt = lds_at<int>(base, C->u);
    N4_LDS int* pu = pt + W0 + 1;
    const int T = uni(pt[W0]);
    if (T < 32 * nch || sizeof(int) * (3 * (size_t)W0 + 4) > uni(C->ubytes)) return false;
    N4_LDS int* ps = pu + W0 + 1;  // [W0 + 1] first strip of every slab, [1] the largest strip
    N4_LDS int* st = ps + W0 + 2;
    // strips of every slab
    for (int x = t; x < W0; x += kResThreads) {
        const int nu = pu[x + 1] - pu[x];
        int n = 0, last = -1;
        UNROLL_4 for (int k = 0; k < nu; ++k) {
            const int strip = (int)(ld_agent(V.res.uent + (size_t)x * V.res.umax + k) & 0xffff) / rows;
            n += strip != last;
            last = strip;
        }
        ps[x] = n;
    }
    if (t == 0) ps[W0 + 1] = 0;
    __syncthreads();
    if (wv == 0) {
        int sum = 0;
        for (int x0 = 0; x0 < W0; x0 += 64) {
            const int n = x0 + lane < W0 ? ps[x0 + lane] : 0;
            int inc = n;
            UNROLL for (int sh = 1; sh < 64; sh <<= 1) {
                const int a = __shfl_up(inc, sh);
                if (lane >= sh) inc += a;
            }
            if (x0 + lane < W0) ps[x0 + lane] = sum + inc - n;
            sum += __shfl(inc, 63);
        }
        if (lane == 0) ps[W0] = sum;
    }
    __syncthreads();
    const int ns = uni(ps[W0]);
    // first tile and first unit of every strip, the waves' cuts and verdicts
    N4_LDS int* su = st + ns + 1;
    N4_LDS int* ok = su + ns + 1;
    N4_LDS uint16_t* cut = reinterpret_cast<N4_LDS uint16_t*>(ok + kResWaves);
    const size_t need = sizeof(int) * (size_t)(3 * W0 + 2 * ns + 6 + kResWaves) + sizeof(uint16_t) * kResWaves * (nch + 1);
    if (ns >= 6 * nch || ns > 0xffff || need > uni(C->ubytes)) return false;
    for (int x = t; x < W0; x += kResThreads) {
        const int nu = pu[x + 1] - pu[x];
        int s = ps[x], last = -1;
        UNROLL_4 for (int k = 0; k < nu; ++k) {
            const uint64_t e = ld_agent(V.res.uent + (size_t)x * V.res.umax + k);
            const int strip = (int)(e & 0xffff) / rows;
            if (strip != last) {
                st[s] = pt[x] + (int)(e >> 48);
                su[s] = pu[x] + k;
                ++s;
            }
            last = strip;
        }
    }
    if (t == 0) {
        st[ns] = T;
        su[ns] = pu[W0];
    }
    __syncthreads();
    for (int i = t; i < ns; i += kResThreads)
        __hip_atomic_fetch_max(ps + W0 + 1, st[i + 1] - st[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __syncthreads();
    const int limit = (T + nch - 1) / nch + uni(ps[W0 + 1]) * (wv + 1) / kResWaves;
    N4_LDS uint16_t* my = cut + wv * (nch + 1);
    int s = 0, k = 0;
    for (; k < nch && s < ns; ++k) {
        if (lane == 0) my[k] = (uint16_t)s;
        const int i = s + lane;
        const unsigned long long fit = __ballot(i < ns && st[i < ns ? i + 1 : ns] - st[s] <= limit);
        const int n = __popcll(fit);
        if (n == 0) break;
        s += n;
    }
    if (lane == 0) ok[wv] = s >= ns;
    for (int i = k + lane; i <= nch; i += 64) my[i] = (uint16_t)ns;
    __syncthreads();
    int w = 0;
    while (w < kResWaves && !uni(ok[w])) ++w;
    if (w == kResWaves) return false;
    N4_LDS int* cb = lds_at<int>(base, C->cb);
    for (int b = c0 + t; b <= c1; b += kResThreads) {
        const int i = cut[w * (nch + 1) + b];
        cb[2 * (b - c0)] = su[i];
        cb[2 * (b - c0) + 1] = st[i];
    }
    return true;
}

// Set-up of a volume: every slab's units (rows of foreground, z ranges) by
// the team's members in turn, the split of the units over the chunks, and
// the packed copy of the own chunks' voxels.  Returns false if the team gave
// up at a barrier.
template <int PREC>
N4_PHASE bool res_setup(const VolDesc* Vp, LdsP smem) {
    const VolDesc& V = *uni(Vp);
    const LdsP base = res_base(smem);
    const CtxP C = res_ctx(base);
    const int rank = uni(C->rank), m = uni(C->m), c0 = uni(C->c0), c1 = uni(C->c1), nb = uni(C->nb);
    N4_LDS int* cb = lds_at<int>(base, C->cb);
    N4_LDS double* red = lds_at<double>(base, C->red);
    const LdsP u = lds_at<unsigned char>(base, C->u);
    const int t = (int)threadIdx.x, wv = uni(t >> 6), lane = t & 63, r16 = lane & 15, g4 = lane >> 4;
    const int W0 = V.W[0], Y = V.W[1], Z = V.W[2];
    const int n = Y * Z;
    uint32_t* team = V.res.team;
    uint64_t* cnt = reinterpret_cast<uint64_t*>(team + kRwMaskWork);
    N4_LDS int* lo = reinterpret_cast<N4_LDS int*>(u);
    N4_LDS int* hi = lo + Y;
    uint32_t count = 0;
    for (int x = rank; x < W0; x += m) {
        for (int y = t; y < Y; y += kResThreads) {
            lo[y] = 0x7fffffff;
            hi[y] = -1;
        }
        __syncthreads();
        const size_t base = (size_t)x * n, q0 = base & ~(size_t)3;
        const int nw = (int)((base + n - q0 + 3) >> 2);
        for (int i = t; i < nw; i += kResThreads) {
            const uint32_t w = *reinterpret_cast<const N4_GLOBAL uint32_t*>(gp(V.wmask) + q0 + 4 * (size_t)i);
            if (!w) continue;
            UNROLL for (int j = 0; j < 4; ++j) {
                const long long v = (long long)(q0 + 4 * (size_t)i + j) - (long long)base;
                if (!((w >> (8 * j)) & 0xffu) || v < 0 || v >= n) continue;
                const int y = (int)fdiv((uint32_t)v, V.mW2), z = (int)v - y * Z;
                __hip_atomic_fetch_min(lo + y, z, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __hip_atomic_fetch_max(hi + y, z, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                ++count;
            }
        }
        __syncthreads();
        if (wv == 0) {
            const int y0 = 16 * lane;
            int zl = 0x7fffffff, zh = -1;
            for (int r = 0; r < 16 && y0 + r < Y; ++r) {
                zl = lo[y0 + r] < zl ? lo[y0 + r] : zl;
                zh = hi[y0 + r] > zh ? hi[y0 + r] : zh;
            }
            const bool on = zh >= 0;
            zl &= ~3;
            const int nt = on ? (zh - zl) / 16 + 1 : 0;
            int inc = nt;
            UNROLL for (int sh = 1; sh < 64; sh <<= 1) {
                const int a = __shfl_up(inc, sh);
                if (lane >= sh) inc += a;
            }
            const unsigned long long live = __ballot(on);
            const int idx = __popcll(live & ((1ull << lane) - 1ull));
            if (on)
                st_agent(V.res.uent + (size_t)x * V.res.umax + idx,
                         (uint64_t)y0 | ((uint64_t)zl << 16) | ((uint64_t)nt << 32) | ((uint64_t)(inc - nt) << 48));
            if (lane == 63)
                st_agent(V.res.slab + x, (uint64_t)__popcll(live) | ((uint64_t)(uint32_t)inc << 32));
        }
        __syncthreads();
    }
    // foreground counts (integers), cleared accumulators
    uint64_t full = 0;
    const int npp = W0 * V.prep_tiles_x;
    for (int i = rank * kResThreads + t; i < npp; i += m * kResThreads) full += (uint64_t)V.ppart[(size_t)4 * i];
    UNROLL for (int sh = 32; sh > 0; sh >>= 1) {
        count += __shfl_xor(count, sh);
        full += __shfl_xor((unsigned long long)full, sh);
    }
    if (lane == 0) {
        if (count) global_add_u64(cnt, count);
        if (full) global_add_u64(cnt + 1, full);
    }
    for (int i = rank * kResThreads + t; i < V.num_copies * V.lmax; i += m * kResThreads)
        st_agent(V.numfx + i, (uint64_t)0);
    for (int i = rank * kResThreads + t; i < V.hist_copies * nb; i += m * kResThreads)
        st_agent(V.hist + i, (uint64_t)0);
    for (int i = t; i < V.lmax; i += kResThreads) lds_at<unsigned long long>(base, C->acc)[i] = 0ull;
    if (!res_barrier(team, m, 0u, smem)) return false;
    // first tile and first unit of every slab
    N4_LDS int* pt = reinterpret_cast<N4_LDS int*>(u);
    N4_LDS int* pu = pt + W0 + 1;
    if (wv == 0) {
        int ct = 0, cu = 0;
        for (int x0 = 0; x0 < W0; x0 += 64) {
            const uint64_t v = x0 + lane < W0 ? ld_agent(V.res.slab + x0 + lane) : 0;
            int it = (int)(v >> 32), iu = (int)(uint32_t)v;
            const int nt = it, nu = iu;
            UNROLL for (int sh = 1; sh < 64; sh <<= 1) {
                const int a = __shfl_up(it, sh), b = __shfl_up(iu, sh);
                if (lane >= sh) {
                    it += a;
                    iu += b;
                }
            }
            if (x0 + lane < W0) {
                pt[x0 + lane] = ct + it - nt;
                pu[x0 + lane] = cu + iu - nu;
            }
            ct += __shfl(it, 63);
            cu += __shfl(iu, 63);
        }
        if (lane == 0) {
            pt[W0] = ct;
            pu[W0] = cu;
        }
    }
    __syncthreads();
    const int T = pt[W0], nch = V.res.nchunk;
    const bool even = res_even_cuts(Vp, smem);
    // else chunk c starts at the first strip whose first tile is >= T c / nchunk
    for (int b = c0 + wv; b <= c1 && !even; b += kResWaves) {
        const int target = (int)((int64_t)T * b / nch);
        int fu = uni(pu[W0]), ft = T;
        if (target < T) {
            int l = 0, h = W0;  // last slab with pt <= target (a slab with tiles)
            while (h - l > 1) {
                const int mid = (l + h) >> 1;
                if (uni(pt[mid]) <= target)
                    l = mid;
                else
                    h = mid;
            }
            const int nu = uni(pu[l + 1]) - uni(pu[l]);
            int s = 0x7fffffff, strip = -1;
            if (lane < nu) {
                const uint64_t e = ld_agent(V.res.uent + (size_t)l * V.res.umax + lane);
                s = pt[l] + (int)(e >> 48);
                strip = (int)(e & 0xffff) / V.wtile_rows;
            }
            const int prev = __shfl_up(strip, 1);
            const unsigned long long ge = __ballot(lane < nu && s >= target && (lane == 0 || prev != strip));
            const int k = ge ? __ffsll(ge) - 1 : nu;
            fu = uni(pu[l]) + k;
            ft = k < nu ? __shfl(s, k) : uni(pt[l + 1]);
        }
        if (lane == 0) {
            cb[2 * (b - c0)] = fu;
            cb[2 * (b - c0) + 1] = ft;
        }
    }
    __syncthreads();
    const int U0 = uni(cb[0]), U1 = uni(cb[2 * (c1 - c0)]);
    float mn = INFINITY, mx = -INFINITY;
    for (int g = U0 + wv; g < U1; g += kResWaves) {
        int l = 0, h = W0;  // last slab with pu <= g (it holds unit g)
        while (h - l > 1) {
            const int mid = (l + h) >> 1;
            if (uni(pu[mid]) <= g)
                l = mid;
            else
                h = mid;
        }
        const uint64_t e = ld_agent(V.res.uent + (size_t)l * V.res.umax + (g - uni(pu[l])));
        const int y0 = uni((int)(e & 0xffff)), zlo = uni((int)((e >> 16) & 0xffff)), nt = uni((int)((e >> 32) & 0xffff));
        const int tile = uni(pt[l]) + uni((int)(e >> 48));
        if (lane == 0) {
            ResUnit r;
            r.x = l;
            r.y0 = (uint16_t)y0;
            r.zlo = (uint16_t)zlo;
            r.tile = tile;
            r.nt = nt;
            V.res.ulist[g] = r;
        }
        const int y = y0 + (PREC == 0 ? 4 * (r16 & 3) + (r16 >> 2) : r16);
        const size_t row = ((size_t)l * Y + (y < Y ? y : 0)) * Z;
        for (int k = 0; k < nt; ++k) {
            const int z = zlo + 16 * k + (PREC == 0 ? g4 : 4 * g4);
            constexpr int zs = PREC == 0 ? 4 : 1;  // z step between a lane's elements
            F4 v = F4{{0.0f, 0.0f, 0.0f, 0.0f}}, cf = v;
            uint32_t mk = 0;
            UNROLL for (int j = 0; j < 4; ++j)
                if (y < Y && z + zs * j < Z) {
                    v.v[j] = gp(V.imlog)[row + z + zs * j];
                    const bool in = gp(V.wmask)[row + z + zs * j] != 0;
                    mk |= in ? 1u << j : 0u;
                    if (V.res.cq) cf.v[j] = gp(V.wconf)[row + z + zs * j];
                    if (in) {
                        mn = fminf(mn, v.v[j]);
                        mx = fmaxf(mx, v.v[j]);
                    }
                }
            const size_t q = (size_t)(tile + k) * 64 + lane;
            store_quad(V.res.xq + 4 * q, v);
            gp(V.res.mq)[q] = (uint8_t)mk;
            if (V.res.cq) store_quad(V.res.cq + 4 * q, cf);
        }
    }
    // the range of the own voxels; the first chunk's partial carries it
    UNROLL for (int sh = 32; sh > 0; sh >>= 1) {
        mn = fminf(mn, __shfl_xor(mn, sh));
        mx = fmaxf(mx, __shfl_xor(mx, sh));
    }
    if (lane == 0) {
        red[2 * wv] = (double)mn;
        red[2 * wv + 1] = (double)mx;
    }
    __syncthreads();
    for (int c = c0 + t; c < c1; c += kResThreads) {
        double a = INFINITY, b = -INFINITY;
        if (c == c0)
            for (int w = 0; w < kResWaves; ++w) {
                a = fmin(a, red[2 * w]);
                b = fmax(b, red[2 * w + 1]);
            }
        double* p = V.res.cpart + 4 * (size_t)c;
        st_agent(p, 0.0);
        st_agent(p + 1, 0.0);
        st_agent(p + 2, a);
        st_agent(p + 3, b);
    }
    return true;
}

// Wiener step of the volume by the workgroup itself: E table and its pairs.
N4_PHASE void res_wiener(const VolDesc* Vp, LdsP smem, double mn, double slope) {
    const LdsP base = res_base(smem);
    const CtxP C = res_ctx(base);
    const int nb = uni(C->nb);
    RunParams rp;
    rp.nbins = nb;
    rp.P = uni(C->P);
    rp.offset = uni(C->offset);
    rp.noise = C->noise;
    rp.fwhm = C->fwhm;
    rp.twiddle = uni(C->twiddle);
    N4_LDS float* E = lds_at<float>(base, C->E);
    wiener_table<kWienerTeam, kResThreads>(*uni(Vp), mn, slope, rp, lds_at<unsigned char>(base, C->u), E);
    __syncthreads();
    N4_LDS float* Ed = lds_at<float>(base, C->Ed);
    for (int i = (int)threadIdx.x; i <= nb; i += kResThreads) {
        const float e = E[i < nb ? i : nb - 1];
        Ed[2 * i] = e;
        Ed[2 * i + 1] = i < nb - 1 ? E[i + 1] - e : 0.0f;
    }
    __syncthreads();
}

// Exact sum of the numerator copies of control point l.
__device__ inline double res_numerator(const uint64_t* numfx, int nc, int lmax, int l) {
    uint64_t c[kResNumCopies];
    UNROLL for (int k = 0; k < kResNumCopies; ++k) c[k] = k < nc ? ld_agent(numfx + (size_t)k * lmax + l) : 0;
    uint64_t s = 0;
    UNROLL for (int k = 0; k < kResNumCopies; ++k) s += c[k];
    return (double)(long long)s / kNumScale;
}

// After the fit: the increment planes of the own slabs; owners update the
// lattice; the histogram copies, read by everyone, are cleared.
N4_PHASE void res_update(LdsP smem, double eps) {
    const LdsP base = res_base(smem);
    const CtxP C = res_ctx(base);
    const int t = (int)threadIdx.x;
    const uint64_t* numfx = uni(C->numfx);
    const double* den = uni(C->den);
    const int nc = uni(C->num_copies), lmax = uni(C->lmax), CyCz = uni(C->Cy) * uni(C->Cz);
    const int l0 = uni(C->pa) * CyCz, n = uni(C->np) * CyCz, o0 = uni(C->o0), o1 = uni(C->o1);
    N4_LDS float* lres = lds_at<float>(base, C->lres);
    for (int e = t; e < n; e += kResThreads) {
        const double d = ld_agent(den + l0 + e);
        lres[e] = (float)(res_numerator(numfx, nc, lmax, l0 + e) / (d + eps));
    }
    double* lat = uni(C->lat);
    for (int l = o0 + t; l < o1; l += kResThreads) {
        const double d = ld_agent(den + l), a = ld_agent(lat + l);
        st_agent(lat + l, a + res_numerator(numfx, nc, lmax, l) / (d + eps));
    }
    uint64_t* hist = uni(C->hist);
    const int nb = uni(C->nb), hc = uni(C->hist_copies), m = uni(C->m);
    for (int k = uni(C->rank); k < hc; k += m)
        for (int i = t; i < nb; i += kResThreads) st_agent(hist + (size_t)k * nb + i, (uint64_t)0);
    __syncthreads();
}

// The numerator copies of the own control points, read by everyone, are
// cleared (den: after their sum has become the level's denominator).
__device__ inline void res_clear_numerator(LdsP base, bool den) {
    const CtxP C = res_ctx(base);
    const int nc = uni(C->num_copies), lmax = uni(C->lmax), o0 = uni(C->o0), o1 = uni(C->o1);
    uint64_t* numfx = uni(C->numfx);
    double* dp = uni(C->den);
    for (int l = o0 + (int)threadIdx.x; l < o1; l += kResThreads) {
        if (den) st_agent(dp + l, res_numerator(numfx, nc, lmax, l));
        for (int k = 0; k < nc; ++k) st_agent(numfx + (size_t)k * lmax + l, (uint64_t)0);
    }
}

// Enters level `level`: refined lattice (owners), tables, denominator.
// False if the team gave up; uses two team barriers from number gen.
template <int PREC>
N4_PHASE bool res_enter_level(const VolDesc* Vp, LdsP smem, int level_, uint32_t gen) {
    const VolDesc& V = *uni(Vp);
    const LdsP base = res_base(smem);
    N4_LDS ResCtx* C = reinterpret_cast<N4_LDS ResCtx*>(base + kResBcBytes);
    const int t = (int)threadIdx.x, level = uni(level_);
    const LevelDesc& LD = V.lev[level];
    const int rank = uni(C->rank), m = uni(C->m), U0 = uni(C->U0), U1 = uni(C->U1);
    uint32_t* team = V.res.team;
    __syncthreads();  // everyone has read the level before
    if (t == 0) {
        for (int d = 0; d < 3; ++d) C->ax[d] = LD.ax[d];
        C->lat = V.lat[level & 1];
        C->Cy = LD.C[1];
        C->Cz = LD.C[2];
        C->L = LD.L;
        C->pa = LD.ax[0][C->x0].b;
        C->np = U1 > U0 ? LD.ax[0][C->x1].b + 4 - C->pa : 0;
        int o0, o1;
        owned_range(LD.L, rank, m, &o0, &o1);
        C->o0 = o0;
        C->o1 = o1;
    }
    __syncthreads();
    res_clear_numerator(base, false);
    const int o0 = uni(C->o0), o1 = uni(C->o1);
    double* lat = uni(C->lat);
    if (level == 0) {
        for (int l = o0 + t; l < o1; l += kResThreads) st_agent(lat + l, 0.0);
    } else {
        if (float* rec = level_lattice_record(V, level - 1)) {
            int p0, p1;
            owned_range(V.lev[level - 1].L, rank, m, &p0, &p1);
            for (int l = p0 + t; l < p1; l += kResThreads) rec[l] = (float)ld_agent(V.lat[(level - 1) & 1] + l);
        }
        for (int l = o0 + t; l < o1; l += kResThreads) st_agent(lat + l, refine_cp<true>(V, level, l));
    }
    const bool single = uni(C->single) != 0;
    res_tables<PREC>(smem, 2);
    if (single) res_load_batch(smem, U0, U1 - U0, 2);
    if (!res_barrier(team, m, gen, smem)) return false;
    res_fit<PREC, true>(smem, 0, 0.0, 1.0);
    if (!res_barrier(team, m, gen + 1, smem)) return false;
    res_clear_numerator(base, true);
    res_tables<PREC>(smem, 1);
    if (single) res_load_batch(smem, U0, U1 - U0, 1);
    __syncthreads();
    return true;
}

// Reconstruction tiles of one volume, if its lattice is ready, while other
// volumes still iterate (run[1] < nvol).
N4_PHASE void res_recon(const VolDesc* Vp, int nvol_, uint32_t* run_, int level, float low, LdsP smem) {
    const VolDesc& V = *uni(Vp);
    const LdsP base = res_base(smem);
    const int nvol = uni(nvol_);
    uint32_t* run = uni(run_);
    uint32_t* team = V.res.team;
    N4_LDS int* bc = reinterpret_cast<N4_LDS int*>(base);
    const int tx = V.recon_tiles_x, rows = V.recon_rows, Y = V.F[1], total = V.F[0] * tx;
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) {
            int tile = -1;
            if (ld_agent(run + 1) < (uint32_t)nvol && ld_agent(team + kRwReady) != 0 &&
                ld_agent(team + kRwTiles) < (uint32_t)total)
                tile = (int)__hip_atomic_fetch_add(team + kRwTiles, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            bc[4] = tile;
        }
        __syncthreads();
        const int tile = uni(bc[4]);
        if (tile < 0 || tile >= total) return;
        const int x = tile / tx, y0 = (tile - x * tx) * rows;
        recon_tile<kResThreads, true>(V, uni(level), low, x, y0, Y - y0 < rows ? Y - y0 : rows, base + kResBcBytes);
    }
}

// One volume, from its set-up to its final lattice, as member `rank` of a
// team of m; false if the team gave up.  ready: count of finished volumes,
// null where no other volume is there to wait for.
template <int PREC>
__device__ bool res_volume(const VolDesc& V, const RunParams& rp, int rank, int m, uint32_t* ready, LdsP smem) {
    const int t = (int)threadIdx.x, wv = uni(t >> 6), lane = t & 63;
    uint32_t* team = V.res.team;
    const int nb = rp.nbins, nch = V.res.nchunk;
    const bool leader = rank == 0;
    N4_LDS ResCtx* C = reinterpret_cast<N4_LDS ResCtx*>(smem + kResBcBytes);
    if (t == 0) {
        ResCtx c;
        carve_res(V, nb, rp.P, PREC, &c);
        c.xq = V.res.xq;
        c.mq = V.res.mq;
        c.cq = V.res.cq;
        c.ulist = V.res.ulist;
        c.numfx = V.numfx;
        c.hist = V.hist;
        c.den = V.den;
        c.lat = V.lat[0];
        c.cpart = V.res.cpart;
        c.Y = V.W[1];
        c.Z = V.W[2];
        c.nbatch = V.res.nbatch;
        c.wtile_rows = V.wtile_rows;
        c.wtiles_x = V.wtiles_x;
        c.num_copies = V.num_copies;
        c.lmax = V.lmax;
        c.hist_copies = V.hist_copies;
        c.nb = nb;
        c.P = rp.P;
        c.offset = rp.offset;
        c.twiddle = rp.twiddle;
        c.fwhm = rp.fwhm;
        c.noise = rp.noise;
        c.nch = nch;
        c.rank = rank;
        c.m = m;
        c.c0 = (int)((int64_t)nch * rank / m);
        c.c1 = (int)((int64_t)nch * (rank + 1) / m);
        *C = c;
    }
    __syncthreads();
    if (!res_setup<PREC>(&V, smem)) return false;
    uint32_t gen = 1;
    __syncthreads();
    if (t == 0) {
        const N4_LDS int* cb = reinterpret_cast<const N4_LDS int*>(smem + C->cb);
        const int k = C->c1 - C->c0;
        C->U0 = cb[0];
        C->T0 = cb[1];
        C->U1 = cb[2 * k];
        C->T1 = cb[2 * k + 1];
        C->single = k == 1 && C->U1 - C->U0 <= C->nbatch;
        C->x0 = C->U1 > C->U0 ? C->ulist[C->U0].x : 0;
        C->x1 = C->U1 > C->U0 ? C->ulist[C->U1 - 1].x : 0;
    }
    N4_LDS unsigned long long* tick = lds_at<unsigned long long>(smem, C->tick);
    N4_LDS double* red = lds_at<double>(smem, C->red);
    if (t < kPhases) tick[t] = 0ull;
    if (!res_barrier(team, m, gen++, smem)) return false;
    VolState* st = V.st;
    const double* cpart = V.res.cpart;
    const uint64_t* cnt = reinterpret_cast<const uint64_t*>(team + kRwMaskWork);
    const uint64_t n_work = ld_agent(cnt), n_full = ld_agent(cnt + 1);
    const double n = (double)n_work;
    int mode = kModeTrans, lvl = 0, it = 0;
    ResTimer pt{tick, leader && V.tphase != nullptr, PhaseTimer::now()};
    for (;;) {
        // partials of the chunks -> range, convergence value, the step's
        // kind.  Up to 64 chunks every wave reduces them itself (no barrier);
        // more go through the waves that hold them and LDS
        const int ops[4] = {0, 0, 1, 2};
        double v[4] = {0.0, 0.0, INFINITY, -INFINITY};
        const bool own = nch <= 64;
        for (int c = own ? lane : t; c < nch; c += own ? 64 : kResThreads) {
            const double* p = cpart + 4 * (size_t)c;
            const double a = ld_agent(p), b = ld_agent(p + 1), d = ld_agent(p + 2), e = ld_agent(p + 3);
            v[0] += a;
            v[1] += b;
            v[2] = fmin(v[2], d);
            v[3] = fmax(v[3], e);
        }
        const int nw = (nch + 63) >> 6;  // waves that hold partials (at most kResWaves: nchunk <= 1024)
        if (own || wv < nw)
            UNROLL for (int sh = 32; sh > 0; sh >>= 1)
                UNROLL for (int k = 0; k < 4; ++k) v[k] = red_apply(ops[k], v[k], __shfl_xor(v[k], sh));
        if (!own) {
            if (wv < nw && lane == 0) UNROLL for (int k = 0; k < 4; ++k) red[4 * wv + k] = v[k];
            __syncthreads();
            UNROLL for (int k = 0; k < 4; ++k) v[k] = red[k];
            for (int w = 1; w < nw; ++w)
                UNROLL for (int k = 0; k < 4; ++k) v[k] = red_apply(ops[k], v[k], red[4 * w + k]);
        }
        const double mn = v[2], mx = v[3];
        double cvv = 0.0;
        int kind = kStepTrans, s_lvl = lvl;
        bool level_end = false;
        if (mode == kModeIter) {
            if (it > 0) cvv = cv_from_sums(v[0], v[1], n);
            const bool stop = it > 0 && !rp.fixed_iters && !(cvv > rp.thr);
            level_end = stop || it >= V.max_iter[lvl];
            if (!level_end) {
                kind = kStepIter;
            } else if (lvl + 1 < rp.nlevels) {
                kind = kStepTrans;
                s_lvl = lvl + 1;
            } else {
                kind = kStepFinal;
            }
        }
        kind = uni(kind);
        s_lvl = uni(s_lvl);
        const double slope = (mx - mn) / (double)(nb - 1);
        const bool degenerate = !(n > 0.0) || !(slope > 0.0);
        if (leader && t == 0) {
            if (mode == kModeIter && it > 0) record_cv(V, lvl, it, cvv);
            if (level_end) {
                st->iters[lvl] = it;
                st->lastcv[lvl] = it > 0 ? cvv : 1e10;
                if (it > 0) st->cv = cvv;
            }
        }
        if (kind == kStepFinal) {
            const double* fin = V.lat[(rp.nlevels - 1) & 1];
            float* rec = level_lattice_record(V, rp.nlevels - 1);
            const int o0 = uni(C->o0), o1 = uni(C->o1);
            for (int l = o0 + t; l < o1; l += kResThreads) {
                const float f = (float)ld_agent(fin + l);
                st_agent(V.latf + l, f);
                if (rec) rec[l] = f;
                if (V.out_lattice) V.out_lattice[l] = f;
            }
            if (leader && t == 0) {
                st->n_mask_full = n_full;
                st->n_mask_work = n_work;
                st->bin_min = mn;
                st->bin_max = mx;
                st->slope = slope;
                st->degenerate = degenerate ? 1 : 0;
                st->mode = kModeFinished;
                st->done = 1;
            }
            if (pt.on && t == 0)
                for (int k = 0; k < kPhases; ++k) V.tphase[k] = tick[k];
            if (ready && !res_barrier(team, m, gen, smem)) return false;
            if (ready && leader && t == 0) {  // the lattice is complete: its reconstruction may start
                st_agent(team + kRwReady, 1u);
                __hip_atomic_fetch_add(ready, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            return true;
        }
        pt.mark(kPhReduce);
        if (pt.on && t == 0) tick[kPhSteps] += 1;
        if (kind == kStepTrans) {
            if (!res_enter_level<PREC>(&V, smem, s_lvl, gen)) return false;
            gen += 2;
            mode = kModeIter;
            lvl = s_lvl;
            it = 0;
            pt.mark(kPhTrans);
            continue;  // (the partials are unchanged)
        }
        // ---- ITER(lvl, it)
        res_clear_numerator(smem, false);
        if (!degenerate) res_hist(smem, mn, slope);
        pt.mark(kPhHist);
        if (!(degenerate ? res_barrier(team, m, gen, smem) : res_barrier_t<true>(team, m, gen, smem, slope))) return false;
        ++gen;
        pt.mark(kPhWait);
        if (!degenerate) res_wiener(&V, smem, mn, slope);
        pt.mark(kPhWiener);
        res_fit<PREC, false>(smem, degenerate, mn, slope);
        pt.mark(kPhFit);
        if (!res_barrier(team, m, gen++, smem)) return false;
        pt.mark(kPhWait);
        res_update(smem, rp.eps);
        pt.mark(kPhUpdate);
        res_eval<PREC>(smem);
        it += 1;
        pt.mark(kPhEval);
        if (!res_barrier(team, m, gen++, smem)) return false;
        pt.mark(kPhWait);
    }
}

}  // namespace n4
#endif
