// eio_resident.h -- time loops that keep a shot's whole state on the chip (k_res_fwd, k_res_adj), and the
// imaging of many coarse samples that the Born passes trade with them through a ring (k_imaging_many).
//
// The launched kernels (eio_kernels.h, eio_step2.h) read two state levels and the media and
// write one or two levels per launch: 50-80 B per cell-update through the caches, and one
// launch per one or two fine steps.  A shot of up to 1.57 M cells (FP64: 0.5 M) fits on the chip: the
// current level in LDS (20 B per FP32 cell of the 160 KB per CU), the older level and the
// media in registers.  Here ONE cooperative launch runs a whole loop: workgroup b owns one
// tile of 64 x TX cells for every fine step, and only the 4-cell halos move, through inboxes in
// device memory.  What is left per step is the stencil itself (VALU and LDS) and the latency
// of one halo exchange.
//
// Exchange.  A wave writes the edge cells of its columns into the neighbours' inboxes as 8-byte
// packets {value, level} with stores that write through to memory (agent-scope cache policy,
// sc1); the receiver reads its inbox with sc1 loads, which miss the caches that are not
// coherent between the 8 XCDs, until every packet carries the level it needs.  A packet is
// one naturally aligned 8-byte access, so it needs no flag, no wait for stores and no cache
// write-back or invalidate: one store and one load of latency per exchange (per-wave
// flags instead cost a store wait, a flag store and a flag poll more: 7.5 us per step of the
// 280 x 472 grid).  Inboxes are double buffered by level parity: a wave sends level k+2 only
// after it has seen its neighbours' level k+1, which they send only after the barrier behind
// their reads of level k.
//
// Hiding the exchange.  A step's edges leave when its level is staged; the next step takes its x
// derivatives first, which need no halo but in the waves at the tile's sides, and asks for
// the halos after them.  The columns along x and their halos are shared out evenly over
// the waves (two each), the rows along z belong to the wave of their columns.
//
// Measured (one launch for the whole loop, FP32): 280 x 472 with R = 1, 3.4 us per fine step
// against 4.0 with two steps per launch; two shots of 520 x 1000 with R = 4, 5.65 us (181
// GCell/s) against 11.2 (92 GCell/s); FP64, two shots of 280 x 472 with R = 2, 6.2 us against 12.2
// with one step per launch.  At R = 4 a step is 14,000 cycles: 1400 the x derivatives, 4700 the z
// derivatives and the update (VALU 383 instructions a wave, LDS 44 words a cell: both about 6500
// cycles of the step when nothing waits), 2000 the staging of the new level, the rest barriers
// and the part of the exchange that the x derivatives do not cover.  Stores that cross the
// fabric cap the exchange at about 3 TB/s (counters of R = 4: 63 % of the wave cycles wait, on the exchange
// and its barriers, 13 % for an issue slot, 24 % issue); neighbours on the same XCD trade through its L2
// (plain stores), which took R = 1 from 4.6 to 3.5 us and R = 4 from 6.4 to 5.85.
//
// Waiting.  All workgroups are co-resident (cooperative launch, at most one workgroup per CU
// by LDS); every wait is bounded by spin_limit polls, after which the workgroup sets *abort
// and leaves, every other workgroup leaves at its next wait, and the host repeats the call with
// the launched kernels (and does not try again for a while).
#pragma once
#include "eio_kernels.h"

namespace eio {

// One tile of a resident loop: rows [z0, z0+64), columns [x0, x0+TX); neighbours' tile
// indices (-1: none); entries of the owned cells, wave by wave (lcell relative to the tile).
constexpr int RES_WX = 16;  // waves of a workgroup
struct ResTile {
    int shot, z0, x0;
    int up, down, left, right;
    int src[RES_WX + 1], rec[RES_WX + 1];
};

constexpr int SC1 = 16;  // cache policy bit of an agent-scope access (write through / miss)

__device__ f32x4_t res_load4(rsrc_t r, int voff, int soff, int aux) __asm("llvm.amdgcn.raw.ptr.buffer.load.v4f32");
__device__ void res_store4(f32x4_t v, rsrc_t r, int voff, int soff, int aux) __asm("llvm.amdgcn.raw.ptr.buffer.store.v4f32");

// A value as 8-byte packets {32 bits, level}: one for float, two for double.
template <typename T>
struct Packet;
template <>
struct Packet<float> {
    static constexpr unsigned BYTES = 8;
    template <int AUX>
    static __device__ __forceinline__ void send(rsrc_t r, float v, int level, unsigned voff, unsigned soff) {
        using u64 = decltype(__builtin_amdgcn_raw_buffer_load_b64(rsrc_t(), 0, 0, 0));
        const unsigned long long p = (unsigned long long)unsigned(level) << 32 | __builtin_bit_cast(unsigned, v);
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u64, p), r, int(voff), int(soff), AUX);
    }
    static __device__ __forceinline__ float value(const f32x4_t* q, int i) { return q[i >> 1][2 * (i & 1)]; }
    static __device__ __forceinline__ bool arrived(const f32x4_t* q, int i, int level) {
        return __builtin_bit_cast(int, float(q[i >> 1][2 * (i & 1) + 1])) == level;
    }
};
template <>
struct Packet<double> {
    static constexpr unsigned BYTES = 16;
    template <int AUX>
    static __device__ __forceinline__ void send(rsrc_t r, double v, int level, unsigned voff, unsigned soff) {
        const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
        f32x4_t p;
        p.x = __builtin_bit_cast(float, unsigned(b));
        p.y = p.w = __builtin_bit_cast(float, level);
        p.z = __builtin_bit_cast(float, unsigned(b >> 32));
        res_store4(p, r, int(voff), int(soff), AUX);
    }
    static __device__ __forceinline__ double value(const f32x4_t* q, int i) {
        const unsigned long long lo = __builtin_bit_cast(unsigned, float(q[i].x)), hi = __builtin_bit_cast(unsigned, float(q[i].z));
        return __builtin_bit_cast(double, hi << 32 | lo);
    }
    static __device__ __forceinline__ bool arrived(const f32x4_t* q, int i, int level) {
        return __builtin_bit_cast(int, float(q[i].y)) == level && __builtin_bit_cast(int, float(q[i].w)) == level;
    }
};

// Four consecutive values of an inbox; only the first `cnt` of them are sent (the others lie
// outside the update region and are zero).
template <typename T>
struct Quad {
    static constexpr int N = int(4 * Packet<T>::BYTES / 16);
    f32x4_t v[N];
    __device__ __forceinline__ void load(rsrc_t r, unsigned voff, unsigned soff) {
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] = res_load4(r, int(voff) + 16 * i, int(soff), SC1);
    }
    __device__ __forceinline__ bool arrived(int cnt, int level) const {
        bool a = true;
#pragma unroll
        for (int i = 0; i < 4; ++i) a = a && (i >= cnt || Packet<T>::arrived(v, i, level));
        return a;
    }
    __device__ __forceinline__ void put(T* dst, int cnt) const {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (i < cnt) dst[i] = Packet<T>::value(v, i);
    }
};

// Inbox of a tile, in values: two level parities of [4 z-fields][halo rows above | below][TX][4]
// and [4 x-fields][halo columns left | right][4][64].
template <int TX>
struct Inbox {
    static constexpr unsigned ZPART = 4u * TX;           // one direction of one field
    static constexpr unsigned XPART = 4u * 64;
    static constexpr unsigned XBASE = 8 * ZPART;
    static constexpr unsigned PARITY = 8 * ZPART + 8 * XPART;
    static constexpr unsigned TILE = 2 * PARITY;
};
// Slots: z-derivative fields vx, vz, szz, sxz and x-derivative fields vx, vz, sxx, sxz.

// The staged levels, addressed from one lane's own cells: an LDS byte address plus an offset,
// added where it is used (an add that the compiler sees would be hoisted out of the time loop,
// one register for each), one address per group of reads within reach of a paired LDS read's 8-bit
// offsets.
template <typename T>
using LdsT = __attribute__((address_space(3))) T;
template <typename T>
__device__ __forceinline__ const LdsT<T>* lds_at(unsigned la, int elem) {
    unsigned a;
    asm volatile("v_add_u32 %0, %2, %1" : "=v"(a) : "v"(la), "i"(elem * int(sizeof(T))));
    return (const LdsT<T>*)a;
}
// D- and D+ along z at row 4 of a window of 9
template <typename T>
__device__ __forceinline__ T dm_l(const LdsT<T>* q, const T* c) {
    return taps<T>(c, q[4] - q[3], q[5] - q[2], q[6] - q[1], q[7] - q[0]);
}
template <typename T>
__device__ __forceinline__ T dp_l(const LdsT<T>* q, const T* c) {
    return taps<T>(c, q[5] - q[4], q[6] - q[3], q[7] - q[2], q[8] - q[1]);
}

// The updates' sums of a forward loop, rounded as the launched loop of the same calls rounds them, so that an NL
// forward gives the same bits in either form: with fused operations spelled out, since which product the compiler
// fuses changes with the code around it.  The free surface's sums, the secondary sources and the adjoint loops are left
// to the compiler: their two forms agree to rounding (an FP32 Born gradient to 5e-7 relative L2).  PAIR (FP32): as k_step2_fwd's streamed stage, variant 12 (d*o first for
// the velocities and, in the second step of a pair, for sxz); else as k_step_fwd.
template <typename T>
__device__ __forceinline__ T fma_t(T a, T b, T c) {
    if constexpr (sizeof(T) == 4) return __builtin_fmaf(a, b, c);
    else return __builtin_fma(a, b, c);
}
template <typename T, bool PAIR>
__device__ __forceinline__ T upd_velocity(T d, T o, T m, T s) {
    return PAIR ? fma_t(m, s, d * o) : fma_t(d, o, m * s);
}
template <typename T>
__device__ __forceinline__ T upd_normal(T d, T o, T mx, T vx, T mz, T vz) {
    return fma_t(d, o, fma_t(mx, vx, mz * vz));
}
template <typename T, bool PAIR>
__device__ __forceinline__ T upd_shear(bool odd, T d, T o, T m, T s) {
    return PAIR && odd ? fma_t(m, s, d * o) : fma_t(d, o, m * s);
}

// The communication of one wave of a tile.
template <typename T, int R>
struct ResComm {
    static constexpr int WX = RES_WX;
    static constexpr int TX = WX * R;
    static constexpr int TXH = TX + 2 * FAT;
    static constexpr unsigned PB = Packet<T>::BYTES;
    static constexpr unsigned NONE = 0x7fff0000u;  // past the end of any inbox
    static constexpr int NZ = (32 * R + 63) / 64;  // z edge stores of a wave
    static constexpr int NQ = R <= 4 ? 1 : 2;      // halo quads of a lane
    using IB = Inbox<TX>;
    rsrc_t box;
    int* abort_flag;
    int spin_limit;
    unsigned zsend[NZ], xsend;  // byte offsets of the lane's edge cells in the neighbours' inboxes (NONE: none)
    int zcell[NZ], xcell;       // and their places in the staged level
    unsigned fetch[NQ];         // byte offsets of the quads the lane reads from its own inbox,
    int cnt[NQ], place[NQ];     // how many of their values are sent, and where they go

    __device__ __forceinline__ void init(const ResTile& t, int tile, int w, int lane, int nz, int nx, T* inbox, unsigned bytes,
                                         int* ab, int* xcd, int spin) {
        static_assert(8 * R + 32 <= 64 * NQ, "quads per lane");
        box = make_rsrc(inbox, bytes);
        abort_flag = ab;
        spin_limit = spin;
        // z edges: item = (field slot, tile above | below, column, row); rows 0..3 become the halo rows
        // below of the tile above, rows 60..63 those above of the one below
#pragma unroll
        for (int i = 0; i < NZ; ++i) {
            const int item = lane + 64 * i, s = item / (8 * R), zi = item % (8 * R);
            const int dn = zi >= 4 * R, c = (zi >> 2) % R, row = zi & 3;
            const int n = dn ? t.down : t.up;
            const bool on = s < 4 && n >= 0 && t.x0 + w * R + c < nx - FAT && (dn || t.z0 + row < nz - FAT);
            zsend[i] = on ? (unsigned(n) * IB::TILE + unsigned(s) * 2 * IB::ZPART + (dn ? 0u : IB::ZPART) +
                             unsigned(w * R + c) * 4 + unsigned(row)) * PB
                          : NONE;
            zcell[i] = (zfield(s & 3) * TXH + FAT + w * R + c) * ZH + FAT + row + (dn ? TZ - FAT : 0);
        }
        // x edges and halos: wave w takes field slot w / 4, side w / 2 % 2 (left, right) and two of its
        // four columns; the left columns become the halo to the right of the tile on the left
        const int s = w >> 2, right = (w >> 1) & 1, c0 = (w & 1) * 2, n = right ? t.right : t.left;
        xsend = n >= 0 && t.z0 + lane < nz - FAT
                    ? (unsigned(n) * IB::TILE + IB::XBASE + unsigned(s) * 2 * IB::XPART + (right ? 0u : IB::XPART) +
                       unsigned(c0) * 64 + unsigned(lane)) * PB
                    : NONE;
        xcell = (xfield(s) * TXH + FAT + (right ? TX - FAT : 0) + c0) * ZH + FAT + lane;
        // quads: the z halo of the wave's columns (8R of them), then its two x halo columns (32)
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
            const int item = lane + 64 * i;
            cnt[i] = 0;
            place[i] = 0;
            unsigned f = 0;
            if (item < 8 * R) {
                const int zs = item / (2 * R), dn = (item / R) & 1, r = item % R;
                if (t.x0 + w * R + r < nx - FAT && (dn ? t.down >= 0 : t.up >= 0)) {
                    cnt[i] = dn ? min(FAT, nz - FAT - (t.z0 + TZ)) : FAT;
                    f = unsigned(zs) * 2 * IB::ZPART + unsigned(dn) * IB::ZPART + unsigned(w * R + r) * 4;
                    place[i] = (zfield(zs) * TXH + FAT + w * R + r) * ZH + (dn ? FAT + TZ : 0);
                }
            } else if (item < 8 * R + 32) {
                const int c = c0 + ((item - 8 * R) >> 4), q = (item - 8 * R) & 15;
                if (n >= 0 && (!right || t.x0 + TX + c < nx - FAT)) {
                    cnt[i] = min(FAT, nz - FAT - (t.z0 + 4 * q));
                    f = IB::XBASE + unsigned(s) * 2 * IB::XPART + (right ? IB::XPART : 0u) + unsigned(c) * 64 + unsigned(q) * 4;
                    place[i] = (xfield(s) * TXH + (right ? FAT + TX : 0) + c) * ZH + FAT + 4 * q;
                }
            }
            fetch[i] = cnt[i] > 0 ? (unsigned(tile) * IB::TILE + f) * PB : NONE;
        }
        // the XCD of this tile and those of its neighbours (each workgroup announces its own)
        unsigned id;
        asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(id));
        const int mine = int(id & 15u) + 1;
        __hip_atomic_store(&xcd[tile], mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int nb = lane == 0 ? t.up : lane == 1 ? t.down : lane == 2 ? t.left : lane == 3 ? t.right : -1;
        int theirs = mine, spins = 0;
        if (nb >= 0)
            while (!(theirs = __hip_atomic_load(&xcd[nb], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
                if (++spins > spin_limit) {
                    __hip_atomic_store(abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    break;
                }
            }
        const bool far_up = __builtin_amdgcn_readlane(theirs, 0) != mine, far_down = __builtin_amdgcn_readlane(theirs, 1) != mine;
        xfar = __builtin_amdgcn_readlane(theirs, right ? 3 : 2) != mine;
#pragma unroll
        for (int i = 0; i < NZ; ++i) zfar[i] = ((lane + 64 * i) % (8 * R)) >= 4 * R ? far_down : far_up;
        // columns of this tile past the grid are not sent
        xcols = right ? 2 : min(2, nx - FAT - (t.x0 + c0));
    }
    int xcols;
    bool zfar[NZ], xfar;   // the receiver is on another XCD
    static __device__ __forceinline__ int zfield(int s) { return s < 2 ? s : s + 1; }
    static __device__ __forceinline__ int xfield(int s) { return s < 3 ? s : 4; }

    // edges of the staged level to the inboxes; pb: byte offset of the level's parity
    __device__ __forceinline__ void send_z(const T* L, int level, unsigned pb) const {
        T v[NZ];
#pragma unroll
        for (int i = 0; i < NZ; ++i) v[i] = L[zcell[i]];
#pragma unroll
        for (int i = 0; i < NZ; ++i)
            if (zsend[i] != NONE) {
                if (zfar[i]) Packet<T>::template send<SC1>(box, v[i], level, zsend[i], pb);
                else Packet<T>::template send<0>(box, v[i], level, zsend[i], pb);
            }
    }
    __device__ __forceinline__ void send_x(const T* L, int level, unsigned pb) const {
        const T a = L[xcell], b = L[xcell + ZH];
        if (xsend != NONE) {
            if (xfar) {
                if (xcols > 0) Packet<T>::template send<SC1>(box, a, level, xsend, pb);
                if (xcols > 1) Packet<T>::template send<SC1>(box, b, level, xsend, pb + 64 * PB);
            } else {
                if (xcols > 0) Packet<T>::template send<0>(box, a, level, xsend, pb);
                if (xcols > 1) Packet<T>::template send<0>(box, b, level, xsend, pb + 64 * PB);
            }
        }
    }
    __device__ __forceinline__ void request(Quad<T> (&q)[NQ], unsigned pb) const {
#pragma unroll
        for (int i = 0; i < NQ; ++i) q[i].load(box, fetch[i], pb);
    }
    __device__ __forceinline__ bool arrived(const Quad<T> (&q)[NQ], int level) const {
        bool a = true;
#pragma unroll
        for (int i = 0; i < NQ; ++i) a = a && q[i].arrived(cnt[i], level);
        return __all(a);
    }
    // the requested halo of `level` into LDS once all of it has arrived; false: gave up
    __device__ __forceinline__ bool receive(Quad<T> (&q)[NQ], T* L, int level, unsigned pb) const {
        int spins = 0;
        while (!arrived(q, level)) {
            if (++spins > spin_limit ||
                ((spins & 63) == 0 && __hip_atomic_load(abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
                __hip_atomic_store(abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return false;
            }
            asm volatile("" ::: "memory");
            request(q, pb);
        }
#pragma unroll
        for (int i = 0; i < NQ; ++i)
            if (cnt[i] > 0) q[i].put(L + place[i], cnt[i]);
        return true;
    }
};

// Fine steps [k0, k1) of the forward loop (a shot stops at its own last step).  MODE: the flags
// of k_step_fwd (F_INJ_COARSE, F_INJ_FINE, F_REC, F_DEC, F_SS: secondary sources from the ring of
// S.sscap coarse samples at S.ss[0], sample j at j % sscap); FSURF: shots with a free surface.
// k0 is a multiple of the shots' sub-sampling.  The state starts from the levels A and B, or from rest
// with from_rest, and goes back there with save, as k_step_fwd finds and leaves it: at an even step A is the
// older level and B the current one, at an odd step (odd sub-samplings) the other way round, so that a
// checkpoint of either form serves both.
template <typename T, int R, int MODE, bool FSURF>
__global__ __launch_bounds__(64 * RES_WX) __attribute__((amdgpu_waves_per_eu(RES_WX / 4, RES_WX / 4)))
void k_res_fwd(const ShotDev<T>* __restrict__ shots, const ResTile* __restrict__ tiles,
               const Entry* __restrict__ ents, T* inbox, unsigned inbox_bytes, int* abort_flag, int* xcd,
               int ntiles, int k0, int k1, int from_rest, int save, int dlo, int dhi, int spin_limit) {
    constexpr int WX = RES_WX;
    constexpr int NT = 64 * WX;
    constexpr int TX = WX * R;
    constexpr int TXH = TX + 2 * FAT;
    constexpr int FS = TXH * ZH;         // values of one staged field
    constexpr unsigned SZ = sizeof(T);
    constexpr bool INJ = (MODE & (F_INJ_COARSE | F_INJ_FINE)) != 0;
    constexpr bool REC = (MODE & F_REC) != 0;
    constexpr bool DEC = (MODE & F_DEC) != 0;
    constexpr bool SS = (MODE & F_SS) != 0;
    constexpr bool PAIR = sizeof(T) == 4 && !FSURF;
    constexpr bool PIN = sizeof(T) == 8 || FSURF || R >= 4;
    // the widest tiles read the media again each step (20 B a cell, from L2) where registers end
    // (R = 5: 7.0 us a step with the media in registers and 10 spilled ones, 7.8 without them)
    constexpr bool NOW = SS && R >= (sizeof(T) == 4 ? 4 : 2);  // nor for a coarse sample on its way
    constexpr bool MEML2 = sizeof(T) == 4 && (R >= 6 || (R >= 5 && DEC) || NOW);
    constexpr int RM = MEML2 ? 1 : R;
    // secondary sources: the coarse sample its in registers, SL fields of its+1 in the LDS that the stage leaves
    constexpr int RS = SS ? R : 1;
    constexpr int SL = !SS ? 0 : sizeof(T) == 4 ? (R <= 3 ? 5 : 3) : (R <= 1 ? 5 : 2);
    __shared__ __attribute__((aligned(16))) T L[5][TXH][ZH];
    __shared__ T LS[SL ? SL : 1][SL ? TX : 1][64];
    __shared__ int s_stop;

    const int tile = xcd_remap(blockIdx.x, ntiles);
    const ResTile& t = tiles[tile];
    const ShotDev<T>& S = shots[t.shot];
    const int nz = S.nz, nx = S.nx, sub = S.sub, h = S.h, nts = S.nts;
    const unsigned n = unsigned(nz) * unsigned(nx);
    const unsigned fbytes = n * SZ, colb = unsigned(nz) * SZ;
    const int kend = min(k1, S.ntw - 1);
    if (k0 >= kend) return;  // the shot (every tile of it) has finished
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int z0 = t.z0, x0 = t.x0;
    const int iz = z0 + lane, zz = lane + FAT;
    const int c0 = FAT + w * R, ix0 = x0 + w * R;
    const unsigned voff = (unsigned(ix0) * unsigned(nz) + unsigned(iz)) * SZ;
    const bool zok = iz < nz - FAT;
    const int ncol = nx - FAT - ix0;     // valid columns of this wave (may exceed R or be negative)
    T cz[4], cx[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) cz[i] = S.cz[i], cx[i] = S.cx[i];
    const T* filt = S.filt;

    if (tid == 0) s_stop = 0;
    T o[5][R], m[5][RM], d[R];
    const rsrc_t rmed = make_rsrc(S.med, 5 * fbytes);
#pragma unroll
    for (int r = 0; r < R; ++r) d[r] = zok && r < ncol ? damp_at(S, iz, ix0 + r) : T(1);
    {
        const rsrc_t rold = make_rsrc((k0 & 1) ? S.B : S.A, 5 * fbytes), rcur = make_rsrc((k0 & 1) ? S.A : S.B, 5 * fbytes);
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int f = 0; f < 5; ++f) {
                const unsigned so = unsigned(r) * colb + unsigned(f) * fbytes;
                if (!MEML2) m[f][MEML2 ? 0 : r] = zok && r < ncol ? bld<T>(rmed, voff, so) : T(0);
                o[f][r] = !from_rest && zok && r < ncol ? bld<T>(rold, voff, so) : T(0);
            }
        for (int e = tid; e < TXH * ZH; e += NT) {
            const int c = e / ZH, z = e - c * ZH;
            const int gx = x0 - FAT + c, gz = z0 - FAT + z;
            const bool in = !from_rest && gx < nx && gz < nz;
            const unsigned vo = in ? (unsigned(gx) * unsigned(nz) + unsigned(gz)) * SZ : 0u;
#pragma unroll
            for (int f = 0; f < 5; ++f) L[f][c][z] = in ? bld<T>(rcur, vo, unsigned(f) * fbytes) : T(0);
        }
    }
    ResComm<T, R> cm;
    cm.init(t, tile, w, lane, nz, nx, inbox, inbox_bytes, abort_flag, xcd, spin_limit);
    // waves whose x derivatives read halo columns
    const bool edge = (w * R < FAT && t.left >= 0) || (w * R + R > TX - FAT && t.right >= 0);
    // the lane's row in the first column of its x window, and 4 rows above its first own cell
    const unsigned lax = unsigned(reinterpret_cast<uintptr_t>((LdsT<T>*)&L[0][c0 - FAT][zz]));
    const unsigned laz = unsigned(reinterpret_cast<uintptr_t>((LdsT<T>*)&L[0][c0][zz - FAT]));

    // the wave's entries: the first 64 are kept in registers, one per lane
    const int sb0 = INJ ? t.src[w] : 0, se0 = INJ ? t.src[w + 1] : 0;
    const int rb0 = REC ? t.rec[w] : 0, re0 = REC ? t.rec[w + 1] : 0;
    const bool fs_top = FSURF && S.surface && z0 == FAT;
    const int its0 = k0 / sub;
    T* const Lf = &L[0][0][0];
    T ra = T(0), rb = T(0);        // receiver sums of samples its, its+1
    int rcell = 0, rrow = -1;      // staged cell, trace row and component
    if (REC && rb0 + lane < re0) {
        const Entry en = ents[rb0 + lane];
        rcell = ((en.crow >> 24) * TXH + FAT + (en.lcell >> 8)) * ZH + FAT + (en.lcell & 255);
        rrow = en.crow;
        const T* tr = S.rec_tr[rrow >> 24] + long(rrow & 0xffffff) * nts;
        ra = tr[its0];
        rb = tr[its0 + 1];
    }
    T sa = T(0), sb = T(0), sd = T(0);  // source samples its, its+1 and the sponge factor
    int scell = 0, srow = -1;
    auto source = [&](int row, int k, int its) -> T {
        if (MODE & F_INJ_FINE) return k < S.ntw ? S.src_tr[row >> 24][long(row & 0xffffff) * S.ntw + k] : T(0);
        return its < nts ? S.src_tr[row >> 24][long(row & 0xffffff) * nts + its] : T(0);
    };
    if (INJ && sb0 + lane < se0) {
        const Entry en = ents[sb0 + lane];
        const int lz = en.lcell & 255, lx = en.lcell >> 8;
        scell = ((en.crow >> 24) * TXH + FAT + lx) * ZH + FAT + lz;
        sd = damp_at(S, z0 + lz, x0 + lx);
        srow = en.crow;
        sa = source(srow, k0, its0);
        sb = source(srow, k0, its0 + 1);
    }
    // decimation sums of the own cells: coarse samples its (xa, za) and its+1 (xb, zb)
    T xa[R], za[R], xb[R], zb[R];
    auto wslot = [&](const T* W, int j) { return make_rsrc(W + size_t(j % S.wcap) * n, fbytes); };
    if constexpr (DEC) {
        const rsrc_t rx = wslot(S.Wvx, its0), rz = wslot(S.Wvz, its0), rx1 = wslot(S.Wvx, its0 + 1), rz1 = wslot(S.Wvz, its0 + 1);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const bool a = its0 != dlo && zok && r < ncol, b = its0 + 1 == dhi && zok && r < ncol;
            xa[r] = a ? bld<T>(rx, voff, unsigned(r) * colb) : T(0);
            za[r] = a ? bld<T>(rz, voff, unsigned(r) * colb) : T(0);
            xb[r] = b ? bld<T>(rx1, voff, unsigned(r) * colb) : T(0);
            zb[r] = b ? bld<T>(rz1, voff, unsigned(r) * colb) : T(0);
        }
    }
    // Vx, Vz of the fine step (js, j2) into the open coarse samples; a complete one is stored
    auto decimate = [&](int js, int j2, const T (&ux)[R], const T (&uz)[R]) {
        const T fa = filt[j2], fb = filt[h + j2];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            xa[r] += ux[r] * fa;
            za[r] += uz[r] * fa;
            xb[r] += ux[r] * fb;
            zb[r] += uz[r] * fb;
        }
        if (j2 == sub) {
            const rsrc_t rx = wslot(S.Wvx, js), rz = wslot(S.Wvz, js);
            const bool acc = js + 2 == dhi;
            const rsrc_t rx2 = wslot(S.Wvx, js + 2), rz2 = wslot(S.Wvz, js + 2);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const unsigned so = unsigned(r) * colb;
                const bool ok = zok && r < ncol;
                if (ok) {
                    bst(rx, xa[r], voff, so);
                    bst(rz, za[r], voff, so);
                }
                xa[r] = xb[r];
                za[r] = zb[r];
                xb[r] = acc && ok ? bld<T>(rx2, voff, so) : T(0);
                zb[r] = acc && ok ? bld<T>(rz2, voff, so) : T(0);
            }
        }
    };
    // secondary sources of the own cells: samples its (gl) and its+1 (gr, fields 0 .. SL-1 in LS), and
    // the next one on its way
    T gl[5][RS], gr[5][RS], gn[5][RS];
    const unsigned las = unsigned(reinterpret_cast<uintptr_t>((LdsT<T>*)&LS[0][SL ? w * R : 0][lane]));
    auto ls = [&](int f, int r) { return const_cast<LdsT<T>*>(lds_at<T>(las, (f * TX + r) * 64)); };
    auto load_ss = [&](int j, T (&u)[5][RS]) {
        const rsrc_t rs = make_rsrc(S.ss[0] + size_t(j % S.sscap) * 5 * n, 5 * fbytes);
#pragma unroll
        for (int r = 0; r < RS; ++r)
#pragma unroll
            for (int f = 0; f < 5; ++f)
                u[f][r] = zok && r < ncol ? bld<T>(rs, voff, unsigned(r) * colb + unsigned(f) * fbytes) : T(0);
    };
    auto take_ss = [&]() {  // gn becomes sample its+1
#pragma unroll
        for (int r = 0; r < RS; ++r)
#pragma unroll
            for (int f = 0; f < 5; ++f) {
                gl[f][r] = f < SL ? T(*ls(f, r)) : gr[f][r];
                if (f < SL) *ls(f, r) = gn[f][r];
                else gr[f][r] = gn[f][r];
            }
    };
    if constexpr (SS) {
        load_ss(its0, gn);
        take_ss();
        load_ss(its0 + 1, gn);
        take_ss();
    }
    constexpr int XG = sizeof(T) == 4 ? 4 : 2;  // columns within reach of one address
    // x derivative D+ / D- of staged field f at the own columns (a register window of R+8);
    // mid: the own values
    auto dx = [&](int f, bool plus, T (&out)[R], T (&mid)[R]) {
        T q[R + 8];
        const LdsT<T>* p = nullptr;
#pragma unroll
        for (int j = 0; j < R + 8; ++j) {
            if (j % XG == 0) p = lds_at<T>(lax, f * FS + j * ZH);
            q[j] = p[(j % XG) * ZH];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            out[r] = plus ? dp_q(q, r + 4, cx) : dm_q(q, r + 4, cx);
            mid[r] = q[r + 4];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) asm volatile("" : "+v"(out[r]));
        if constexpr (PIN) __builtin_amdgcn_sched_barrier(0);
    };
    T dxx[R], dxz[R], vxx[R], vzx[R];   // x derivatives of sxx, sxz, vx, vz
    auto dx_all = [&](int js, int j2) {
        T ux[R], uz[R], mid[R];
        dx(2, false, dxx, mid);
        dx(4, true, dxz, mid);
        dx(0, true, vxx, ux);
        dx(1, false, vzx, uz);
        // the staged velocities are the result of the step before: their decimation rides along
        if constexpr (DEC) {
            if (js >= 0) decimate(js, j2, ux, uz);
        }
    };
    // z derivatives and the update: the next level into o
    T mnext[5];
    auto load_media = [&](int r) {
#pragma unroll
        for (int f = 0; f < 5; ++f) mnext[f] = zok && r < ncol ? bld<T>(rmed, voff, unsigned(r) * colb + unsigned(f) * fbytes) : T(0);
    };
    auto update = [&](bool odd, T fl, T fr) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            T mm[5];
#pragma unroll
            for (int f = 0; f < 5; ++f) mm[f] = MEML2 ? mnext[f] : m[f][MEML2 ? 0 : r];
            if (MEML2 && r + 1 < R) load_media(r + 1);
            const T s0 = dxx[r] + dp_l(lds_at<T>(laz, 4 * FS + r * ZH), cz);
            const T s1 = dm_l(lds_at<T>(laz, 3 * FS + r * ZH), cz) + dxz[r];
            const T vzz = dp_l(lds_at<T>(laz, FS + r * ZH), cz);
            const T sh = dm_l(lds_at<T>(laz, r * ZH), cz) + vzx[r];
            T a0, a1, a2, a3, a4;
            if (!FSURF || !fs_top) {
                a0 = upd_velocity<T, PAIR>(d[r], o[0][r], mm[0], s0);
                a1 = upd_velocity<T, PAIR>(d[r], o[1][r], mm[1], s1);
                a2 = upd_normal<T>(d[r], o[2][r], mm[2], vxx[r], mm[3], vzz);
                a3 = upd_normal<T>(d[r], o[3][r], mm[3], vxx[r], mm[2], vzz);
                a4 = upd_shear<T, PAIR>(odd, d[r], o[4][r], mm[4], sh);
            } else {  // kernelsGpuElastic.cu:589-776, as in k_step_fwd
                const bool on = iz == SURF, below = iz > SURF;
                a0 = d[r] * o[0][r] + ((on || below) ? mm[0] * s0 : T(0));
                a1 = d[r] * o[1][r] + (below ? mm[1] * s1 : T(0));
                a2 = d[r] * o[2][r] + (below ? (mm[2] * vxx[r] + mm[3] * vzz)
                                             : (on ? (mm[2] - mm[3] * mm[3] / mm[2]) * vxx[r] : T(0)));
                a3 = d[r] * o[3][r] + (below ? (mm[3] * vxx[r] + mm[2] * vzz) : T(0));
                a4 = d[r] * o[4][r] + (below ? mm[4] * sh : T(0));
            }
            if constexpr (SS) {  // secondary source sampled at it2-1 (kernelsGpuElastic.cu:1363-1368)
                T* const a[5] = {&a0, &a1, &a2, &a3, &a4};
#pragma unroll
                for (int f = 0; f < 5; ++f) *a[f] += gl[f][r] * fl + (f < SL ? T(*ls(f, r)) : gr[f][r]) * fr;
            }
            o[0][r] = d[r] * a0;
            o[1][r] = d[r] * a1;
            o[2][r] = d[r] * a2;
            o[3][r] = d[r] * a3;
            o[4][r] = d[r] * a4;
            // one column at a time where the registers are short
            if constexpr (PIN) {
#pragma unroll
                for (int f = 0; f < 5; ++f) asm volatile("" : "+v"(o[f][r]));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    __syncthreads();

    constexpr unsigned PARITY = Inbox<TX>::PARITY * Packet<T>::BYTES;
    int its = its0, it2 = 0;      // fine step k = its*sub + it2
    int js = -1, j2 = 0;          // the step before k: it2 counted from 1
    for (int k = k0; k < kend; ++k) {
        const unsigned pr = (unsigned(k) & 1u) * PARITY;
        Quad<T> q[ResComm<T, R>::NQ];
        if (k > k0) cm.send_x(Lf, k, pr);
        if constexpr (SS)
            if (!NOW && k > k0 && it2 == 0) take_ss();
        if (!edge) dx_all(js, j2);
        if (k > k0) {
            cm.request(q, pr);
            if (!cm.receive(q, Lf, k, pr)) s_stop = 1;
        }
        __syncthreads();  // the halos are staged
        if (s_stop) return;
        if (MEML2) load_media(0);
        if (edge) dx_all(js, j2);
        update(k & 1, SS ? filt[it2] : T(0), SS ? filt[h + it2] : T(0));
        __syncthreads();  // every read of level k is done
        // the next level is staged, this one becomes the older one; what follows touches the
        // wave's own columns only, and the LDS accesses of one wave are in order
        if (zok) {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (r < ncol) {
                    LdsT<T>* p = const_cast<LdsT<T>*>(lds_at<T>(laz, r * ZH + FAT));
#pragma unroll
                    for (int f = 0; f < 5; ++f) {
                        const T c = p[f * FS];
                        p[f * FS] = o[f][r];
                        o[f][r] = c;
                    }
                    if constexpr (PIN) __builtin_amdgcn_sched_barrier(0);
                }
        }
        __builtin_amdgcn_wave_barrier();
        if (INJ && sb0 < se0) {
            const T fa = filt[it2], fb = filt[h + it2];
            if (srow >= 0) {
                Lf[scell] = mac(T(Lf[scell]), sd, (MODE & F_INJ_FINE) ? sa : mul2(sa, fa, sb, fb));
                if (MODE & F_INJ_FINE) {
                    sa = source(srow, k + 1, 0);
                } else if (it2 + 1 == sub) {
                    sa = sb;
                    sb = source(srow, 0, its + 2);
                }
            }
            for (int e = sb0 + 64 + lane; e < se0; e += 64) {
                const Entry en = ents[e];
                const int lz = en.lcell & 255, lx = en.lcell >> 8;
                const T s = (MODE & F_INJ_FINE) ? source(en.crow, k, 0) : mul2(source(en.crow, 0, its), fa, source(en.crow, 0, its + 1), fb);
                T& v = L[en.crow >> 24][FAT + lx][FAT + lz];
                v = mac(v, damp_at(S, z0 + lz, x0 + lx), s);
            }
            __builtin_amdgcn_wave_barrier();
        }
        js = its;
        j2 = it2 + 1;
        if (REC && rb0 < re0) {
            const T fa = filt[j2], fb = filt[h + j2];
            if (rrow >= 0) {
                const T v = Lf[rcell];
                ra = mac(ra, v, fa);
                rb = mac(rb, v, fb);
                if (j2 == sub) {
                    S.rec_tr[rrow >> 24][long(rrow & 0xffffff) * nts + js] = ra;
                    ra = rb;
                    rb = T(0);
                }
            }
            for (int e = rb0 + 64 + lane; e < re0; e += 64) {
                const Entry en = ents[e];
                const T v = L[en.crow >> 24][FAT + (en.lcell >> 8)][FAT + (en.lcell & 255)];
                T* tr = S.rec_tr[en.crow >> 24] + long(en.crow & 0xffffff) * nts + js;
                tr[0] = mac(tr[0], v, fa);
                tr[1] = mac(tr[1], v, fb);
            }
            __builtin_amdgcn_wave_barrier();
        }
        if (FSURF && fs_top && lane <= FAT) {  // the free-surface map (fs_map_col) of the own columns
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (r < ncol) {
                    T* p = Lf + (c0 + r) * ZH;   // row zz = lane + 4, the surface is row 8
                    const T szz = p[3 * FS + 2 * SURF - zz], sxz = p[4 * FS + 2 * SURF + 1 - zz];
                    if (lane < FAT) p[zz] = T(0);
                    p[FS + zz] = T(0);
                    p[3 * FS + zz] = lane < FAT ? -szz : T(0);
                    if (lane > 0) p[4 * FS + zz] = -sxz;
                }
            __builtin_amdgcn_wave_barrier();
        }
        if constexpr (SS)
            if (it2 + 1 == sub && k + 1 < kend) {
                load_ss(its + 2, gn);
                if (NOW) take_ss();
            }
        if (k + 1 < kend) cm.send_z(Lf, k + 1, PARITY - pr);
        if (++it2 == sub) {
            it2 = 0;
            ++its;
        }
        __syncthreads();  // the next level is staged
    }
    // the open sums; the last step's decimation; the state
    if (REC && rrow >= 0) {
        T* tr = S.rec_tr[rrow >> 24] + long(rrow & 0xffffff) * nts;
        tr[its] = ra;
        if (it2) tr[its + 1] = rb;
    }
    if constexpr (DEC) {
        T ux[R], uz[R];
#pragma unroll
        for (int r = 0; r < R; ++r) ux[r] = L[0][c0 + r][zz], uz[r] = L[1][c0 + r][zz];
        decimate(js, j2, ux, uz);
        const rsrc_t rx = wslot(S.Wvx, its), rz = wslot(S.Wvz, its);
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (zok && r < ncol) {
                bst(rx, xa[r], voff, unsigned(r) * colb);
                bst(rz, za[r], voff, unsigned(r) * colb);
            }
    }
    if (save) {
        const rsrc_t rold = make_rsrc((kend & 1) ? S.B : S.A, 5 * fbytes), rcur = make_rsrc((kend & 1) ? S.A : S.B, 5 * fbytes);
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (zok && r < ncol) {
#pragma unroll
                for (int f = 0; f < 5; ++f) {
                    const unsigned so = unsigned(r) * colb + unsigned(f) * fbytes;
                    bst(rold, o[f][r], voff, so);
                    bst(rcur, L[f][c0 + r][zz], voff, so);
                }
            }
    }
}

// Reverse fine steps [k0, k1) of the adjoint loop.  MODE M_NLADJ: the NL adjoint (source traces
// extracted); M_BADJ: the Born receiver pass, whose adjoint fields of a coarse sample are summed in
// registers and stored once, complete, into the ring of S.sscap samples at S.ss[0] (sample j at j %
// sscap); a launch that ends above sample 0 leaves the open sample there for the next one.  k0 and,
// for M_BADJ, k1 are multiples of the sub-sampling.  The stage holds the media-scaled level (as
// k_step_adj), so the current level itself stays in registers with the older one.  Bound as the
// forward loop is (a step of R = 4 with the media from L2 where registers end); two shots of 520 x
// 1000, R = 4, 5.9 us a reverse step against 17.2 with two steps per launch, 280 x 472, R = 1, 3.35
// against 4.7, and FP64, two of 280 x 472, R = 2, 7.65 against 12.0.  The receiver pass (with the source
// pass and the imaging): 600 x 1592, R = 4, 16.5 against 35.4 (19.4 with the media from L2 and every x
// derivative held over the exchange, 34 registers spilled; 17.6 with the derivatives one field at a time);
// four of 280 x 472, R = 3, 12.3 against 24.3.
template <typename T, int R, int MODE>
__global__ __launch_bounds__(64 * RES_WX) __attribute__((amdgpu_waves_per_eu(RES_WX / 4, RES_WX / 4)))
void k_res_adj(const ShotDev<T>* __restrict__ shots, const ResTile* __restrict__ tiles,
               const Entry* __restrict__ ents, T* inbox, unsigned inbox_bytes, int* abort_flag, int* xcd,
               int ntiles, int k0, int k1, int from_rest, int save, int spin_limit) {
    constexpr int WX = RES_WX;
    constexpr int NT = 64 * WX;
    constexpr int TX = WX * R;
    constexpr int TXH = TX + 2 * FAT;
    constexpr int FS = TXH * ZH;
    constexpr unsigned SZ = sizeof(T);
    constexpr bool BORN = MODE == M_BADJ;
    // where registers end: the receiver pass takes its x derivatives one field at a time behind the halos
    // and keeps ML media fields in the LDS that the stage leaves; the NL adjoint reads the media again each
    // step (from L2)
    constexpr bool WIDE = BORN && R >= (sizeof(T) == 4 ? 4 : 2);
    constexpr int ML = !WIDE ? 0 : sizeof(T) == 4 ? 3 : 2;
    constexpr bool MEML2 = !BORN && sizeof(T) == 4 && R >= 5;
    constexpr int RM = MEML2 ? 1 : R;
    constexpr int RB = BORN ? R : 1;
    constexpr bool PIN = sizeof(T) == 8 || R >= 3;
    __shared__ __attribute__((aligned(16))) T L[5][TXH][ZH];
    __shared__ T LM[ML ? ML : 1][ML ? TX : 1][64];
    __shared__ int s_stop;

    const int tile = xcd_remap(blockIdx.x, ntiles);
    const ResTile& t = tiles[tile];
    const ShotDev<T>& S = shots[t.shot];
    const int nz = S.nz, nx = S.nx, sub = S.sub, h = S.h, nts = S.nts;
    const unsigned n = unsigned(nz) * unsigned(nx);
    const unsigned fbytes = n * SZ, colb = unsigned(nz) * SZ;
    const int kend = min(k1, S.ntw - 1);
    if (k0 >= kend) return;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int z0 = t.z0, x0 = t.x0;
    const int iz = z0 + lane, zz = lane + FAT;
    const int c0 = FAT + w * R, ix0 = x0 + w * R;
    const unsigned voff = (unsigned(ix0) * unsigned(nz) + unsigned(iz)) * SZ;
    const bool zok = iz < nz - FAT;
    const int ncol = nx - FAT - ix0;
    T cz[4], cx[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) cz[i] = S.cz[i], cx[i] = S.cx[i];
    const T* filt = S.filt;

    if (tid == 0) s_stop = 0;
    T o[5][R], c[5][R], m[5][RM], d[R];   // older and current level, media, sponge of the own cells
    const rsrc_t rmed = make_rsrc(S.med, 5 * fbytes);
#pragma unroll
    for (int r = 0; r < R; ++r) d[r] = zok && r < ncol ? damp_at(S, iz, ix0 + r) : T(1);
    {
        const rsrc_t rold = make_rsrc(S.A, 5 * fbytes), rcur = make_rsrc(S.B, 5 * fbytes);
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int f = 0; f < 5; ++f) {
                const unsigned so = unsigned(r) * colb + unsigned(f) * fbytes;
                const bool ok = zok && r < ncol;
                const T mf = !MEML2 && ok ? bld<T>(rmed, voff, so) : T(0);
                if (f < ML) LM[f < ML ? f : 0][ML ? w * R + r : 0][lane] = mf;
                else if (!MEML2) m[f][MEML2 ? 0 : r] = mf;
                o[f][r] = !from_rest && ok ? bld<T>(rold, voff, so) : T(0);
                c[f][r] = !from_rest && ok ? bld<T>(rcur, voff, so) : T(0);
            }
        for (int e = tid; e < TXH * ZH; e += NT) {
            const int cc = e / ZH, z = e - cc * ZH;
            const int gx = x0 - FAT + cc, gz = z0 - FAT + z;
            const bool in = !from_rest && gx < nx && gz < nz;
            const unsigned vo = in ? (unsigned(gx) * unsigned(nz) + unsigned(gz)) * SZ : 0u;
            T u[5], g[5];
#pragma unroll
            for (int f = 0; f < 5; ++f) {
                u[f] = in ? bld<T>(rcur, vo, unsigned(f) * fbytes) : T(0);
                g[f] = in ? bld<T>(rmed, vo, unsigned(f) * fbytes) : T(0);
            }
            L[0][cc][z] = g[0] * u[0];
            L[1][cc][z] = g[1] * u[1];
            L[2][cc][z] = g[2] * u[2] + g[3] * u[3];
            L[3][cc][z] = g[3] * u[2] + g[2] * u[3];
            L[4][cc][z] = g[4] * u[4];
        }
    }
    ResComm<T, R> cm;
    cm.init(t, tile, w, lane, nz, nx, inbox, inbox_bytes, abort_flag, xcd, spin_limit);
    const bool edge = (w * R < FAT && t.left >= 0) || (w * R + R > TX - FAT && t.right >= 0);
    const unsigned lax = unsigned(reinterpret_cast<uintptr_t>((LdsT<T>*)&L[0][c0 - FAT][zz]));
    const unsigned lam = unsigned(reinterpret_cast<uintptr_t>((LdsT<T>*)&LM[0][ML ? w * R : 0][lane]));
    const unsigned laz = unsigned(reinterpret_cast<uintptr_t>((LdsT<T>*)&L[0][c0][zz - FAT]));

    // the wave's entries (data to inject, source cells to read), the first 64 of each in registers
    const int rb0 = t.rec[w], re0 = t.rec[w + 1];
    const int sb0 = BORN ? 0 : t.src[w], se0 = BORN ? 0 : t.src[w + 1];
    const bool entries = rb0 < re0 || sb0 < se0;
    int its = nts - 2 - k0 / sub, it2 = sub - 1;   // as adj_time; k0 is a multiple of sub
    T* const Lf = &L[0][0][0];
    auto sample = [&](int row, int j) -> T {
        return j >= 0 ? S.rec_tr[row >> 24][long(row & 0xffffff) * nts + j] : T(0);
    };
    T ra = T(0), rb = T(0), rd = T(0);   // data samples its, its+1, sponge factor
    int rcell = 0, rrow = -1;
    if (rb0 + lane < re0) {
        const Entry en = ents[rb0 + lane];
        const int lz = en.lcell & 255, lx = en.lcell >> 8;
        rcell = ((en.crow >> 24) * TXH + FAT + lx) * ZH + FAT + lz;
        rd = damp_at(S, z0 + lz, x0 + lx);
        rrow = en.crow;
        ra = sample(rrow, its);
        rb = sample(rrow, its + 1);
    }
    T sa = T(0), sb = T(0);              // source-trace sums of samples its, its+1
    int scell = 0, srow = -1;
    auto strace = [&](int row) -> T* { return S.src_tr[row >> 24] + long(row & 0xffffff) * nts; };
    if (!BORN && sb0 + lane < se0) {
        const Entry en = ents[sb0 + lane];
        scell = ((en.crow >> 24) * TXH + FAT + (en.lcell >> 8)) * ZH + FAT + (en.lcell & 255);
        srow = en.crow;
        sb = strace(srow)[its + 1];
    }
    // adjoint fields of the own cells: coarse samples its+1 (ax) and its (ay)
    T ax[5][RB], ay[5][RB];
    auto slot = [&](int j) { return make_rsrc(S.ss[0] + size_t(j % S.sscap) * 5 * n, 5 * fbytes); };
    auto store_slot = [&](int j) {
        const rsrc_t rs = slot(j);
        if (zok) {
#pragma unroll
            for (int r = 0; r < RB; ++r)
                if (r < ncol) {
#pragma unroll
                    for (int f = 0; f < 5; ++f) bst(rs, ax[f][r], voff, unsigned(r) * colb + unsigned(f) * fbytes);
                }
        }
    };
    if constexpr (BORN) {
        const rsrc_t rs = slot(its + 1);
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int f = 0; f < 5; ++f) {
                ax[f][r] = !from_rest && zok && r < ncol ? bld<T>(rs, voff, unsigned(r) * colb + unsigned(f) * fbytes) : T(0);
                ay[f][r] = T(0);
            }
    }
    constexpr int XG = sizeof(T) == 4 ? 4 : 2;
    auto dx = [&](int f, bool plus, T (&out)[R]) {
        T q[R + 8];
        const LdsT<T>* p = nullptr;
#pragma unroll
        for (int j = 0; j < R + 8; ++j) {
            if (j % XG == 0) p = lds_at<T>(lax, f * FS + j * ZH);
            q[j] = p[(j % XG) * ZH];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) out[r] = plus ? dp_q(q, r + 4, cx) : dm_q(q, r + 4, cx);
#pragma unroll
        for (int r = 0; r < R; ++r) asm volatile("" : "+v"(out[r]));
        if constexpr (PIN) __builtin_amdgcn_sched_barrier(0);
    };
    T dxa[R], dx6[R], dx0[R], dx1[R];   // x derivatives of the stage's fields 2, 4, 0, 1
    auto dx_all = [&]() {
        dx(2, false, dxa);
        dx(4, true, dx6);
        dx(0, true, dx0);
        dx(1, false, dx1);
    };
    T mnext[5];
    auto load_media = [&](int r) {
#pragma unroll
        for (int f = 0; f < 5; ++f) mnext[f] = zok && r < ncol ? bld<T>(rmed, voff, unsigned(r) * colb + unsigned(f) * fbytes) : T(0);
    };
    __syncthreads();

    constexpr unsigned PARITY = Inbox<TX>::PARITY * Packet<T>::BYTES;
    for (int k = k0; k < kend; ++k) {
        const unsigned pr = (unsigned(k) & 1u) * PARITY;
        Quad<T> q[ResComm<T, R>::NQ];
        if (k > k0) cm.send_x(Lf, k, pr);
        if (!WIDE && !edge) dx_all();
        if (k > k0) {
            cm.request(q, pr);
            if (!cm.receive(q, Lf, k, pr)) s_stop = 1;
        }
        __syncthreads();  // the halos are staged
        if (s_stop) return;
        if (!WIDE && edge) dx_all();
        // the next level into o, which trades places with the current one
        if constexpr (WIDE) {
            T x[R];
            auto next = [&](int f, int r, T sum) {
                const T v = d[r] * (d[r] * o[f][r] - sum);
                o[f][r] = c[f][r];
                c[f][r] = v;
                asm volatile("" : "+v"(c[f][r]), "+v"(o[f][r]));
            };
            dx(2, false, x);
#pragma unroll
            for (int r = 0; r < R; ++r) next(0, r, x[r] + dp_l(lds_at<T>(laz, 4 * FS + r * ZH), cz));
            dx(4, true, x);
#pragma unroll
            for (int r = 0; r < R; ++r) next(1, r, dm_l(lds_at<T>(laz, 3 * FS + r * ZH), cz) + x[r]);
            dx(0, true, x);
#pragma unroll
            for (int r = 0; r < R; ++r) next(2, r, x[r]);
#pragma unroll
            for (int r = 0; r < R; ++r) next(3, r, dp_l(lds_at<T>(laz, FS + r * ZH), cz));
            dx(1, false, x);
#pragma unroll
            for (int r = 0; r < R; ++r) next(4, r, dm_l(lds_at<T>(laz, r * ZH), cz) + x[r]);
        } else {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const T d6 = dp_l(lds_at<T>(laz, 4 * FS + r * ZH), cz);
            const T db = dm_l(lds_at<T>(laz, 3 * FS + r * ZH), cz);
            const T d1 = dp_l(lds_at<T>(laz, FS + r * ZH), cz);
            const T d0 = dm_l(lds_at<T>(laz, r * ZH), cz);
            T v[5];
            v[0] = d[r] * (d[r] * o[0][r] - (dxa[r] + d6));
            v[1] = d[r] * (d[r] * o[1][r] - (db + dx6[r]));
            v[2] = d[r] * (d[r] * o[2][r] - dx0[r]);
            v[3] = d[r] * (d[r] * o[3][r] - d1);
            v[4] = d[r] * (d[r] * o[4][r] - (d0 + dx1[r]));
#pragma unroll
            for (int f = 0; f < 5; ++f) {
                o[f][r] = c[f][r];
                c[f][r] = v[f];
            }
            if constexpr (PIN) {
#pragma unroll
                for (int f = 0; f < 5; ++f) asm volatile("" : "+v"(c[f][r]), "+v"(o[f][r]));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        }
        if (MEML2) load_media(0);
        __syncthreads();  // every read of level k is done
        if (entries) {  // through the wave's own columns: data into the new level, source cells out of it
            if (zok) {
#pragma unroll
                for (int r = 0; r < R; ++r)
                    if (r < ncol) {
                        LdsT<T>* p = const_cast<LdsT<T>*>(lds_at<T>(laz, r * ZH + FAT));
#pragma unroll
                        for (int f = 0; f < 5; ++f) p[f * FS] = c[f][r];
                    }
            }
            __builtin_amdgcn_wave_barrier();
            if (rb0 < re0) {
                const T fa = filt[it2 + 1], fb = filt[h + it2 + 1];
                if (rrow >= 0) {
                    Lf[rcell] += rd * (ra * fa + rb * fb);
                    if (it2 == 0) {
                        rb = ra;
                        ra = sample(rrow, its - 1);
                    }
                }
                for (int e = rb0 + 64 + lane; e < re0; e += 64) {
                    const Entry en = ents[e];
                    const int lz = en.lcell & 255, lx = en.lcell >> 8;
                    const T s = sample(en.crow, its) * fa + sample(en.crow, its + 1) * fb;
                    L[en.crow >> 24][FAT + lx][FAT + lz] += damp_at(S, z0 + lz, x0 + lx) * s;
                }
                __builtin_amdgcn_wave_barrier();
                if (zok) {
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        if (r < ncol) {
                            const LdsT<T>* p = lds_at<T>(laz, r * ZH + FAT);
#pragma unroll
                            for (int f = 0; f < 5; ++f) c[f][r] = p[f * FS];
                        }
                }
            }
            if (!BORN && sb0 < se0) {
                const T fa = filt[it2], fb = filt[h + it2];
                if (srow >= 0) {
                    const T v = Lf[scell];
                    sa += v * fa;
                    sb += v * fb;
                    if (it2 == 0) {
                        strace(srow)[its + 1] = sb;
                        sb = sa;
                        sa = T(0);
                    }
                }
                for (int e = sb0 + 64 + lane; e < se0; e += 64) {
                    const Entry en = ents[e];
                    const T v = L[en.crow >> 24][FAT + (en.lcell >> 8)][FAT + (en.lcell & 255)];
                    T* tr = strace(en.crow) + its;
                    tr[0] += v * fa;
                    tr[1] += v * fb;
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
        // the scaled next level is staged
#pragma unroll
        for (int r = 0; r < R; ++r) {
            T g[5];
#pragma unroll
            for (int f = 0; f < 5; ++f)
                g[f] = f < ML ? T(*lds_at<T>(lam, (f * TX + r) * 64)) : MEML2 ? mnext[f] : m[f][MEML2 ? 0 : r];
            if (MEML2 && r + 1 < R) load_media(r + 1);
            if (zok && r < ncol) {
                LdsT<T>* p = const_cast<LdsT<T>*>(lds_at<T>(laz, r * ZH + FAT));
                p[0] = g[0] * c[0][r];
                p[FS] = g[1] * c[1][r];
                p[2 * FS] = g[2] * c[2][r] + g[3] * c[3][r];
                p[3 * FS] = g[3] * c[2][r] + g[2] * c[3][r];
                p[4 * FS] = g[4] * c[4][r];
            }
            if constexpr (PIN) __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_wave_barrier();
        if (k + 1 < kend) cm.send_z(Lf, k + 1, PARITY - pr);
        if constexpr (BORN) {
            const T ea = filt[it2], eb = filt[h + it2];
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int f = 0; f < 5; ++f) {
                    ay[f][r] += c[f][r] * ea;
                    ax[f][r] += c[f][r] * eb;
                }
            if (it2 == 0) {
                store_slot(its + 1);
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int f = 0; f < 5; ++f) {
                        ax[f][r] = ay[f][r];
                        ay[f][r] = T(0);
                    }
            }
        }
        if (--it2 < 0) {
            it2 = sub - 1;
            --its;
        }
        __syncthreads();  // the next level is staged
    }
    // the open sums and the state (its, it2: the step after the last one)
    if (!BORN && srow >= 0) {
        T* tr = strace(srow);
        tr[its + 1] = sb;
        if (it2 != sub - 1) tr[its] = sa;
    }
    if constexpr (BORN) store_slot(its + 1);
    if (save) {
        const rsrc_t rold = make_rsrc(S.A, 5 * fbytes), rcur = make_rsrc(S.B, 5 * fbytes);
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (zok && r < ncol) {
#pragma unroll
                for (int f = 0; f < 5; ++f) {
                    const unsigned so = unsigned(r) * colb + unsigned(f) * fbytes;
                    bst(rold, o[f][r], voff, so);
                    bst(rcur, c[f][r], voff, so);
                }
            }
    }
}

// ------------------------------------------------------------------ imaging over many coarse samples
// k_imaging for coarse samples j0, j0 - 1, .., j1 (ADJ: the imaging condition with the ring's adjoint
// fields) or j0, j0 + 1, .., j1 (forward: the secondary sources into the ring), sample j at j % sscap
// of S.ss[0].  The perturbation or the accumulators stay in registers over the samples, and the
// slices next to a sample are in L2 from its neighbours' turn: 31 B a cell and sample instead of 104 (ADJ).
template <typename T, int R, int WX, bool ADJ>
__global__ __launch_bounds__(64 * WX) void k_imaging_many(const ShotDev<T>* __restrict__ shots,
                                                          const TileDev* __restrict__ tiles, int ntiles, int j0, int j1) {
    if (!ADJ) {  // the samples are independent: the grid's y direction shares them out
        const int per = (j1 - j0 + int(gridDim.y)) / int(gridDim.y);
        j0 += int(blockIdx.y) * per;
        j1 = min(j1, j0 + per - 1);
        if (j0 > j1) return;
    }
    constexpr int NT = 64 * WX;
    constexpr int TX = WX * R;
    constexpr int TXH = TX + 2 * FAT;
    constexpr unsigned SZ = sizeof(T);
    constexpr int NFILL = (TXH * ZH + NT - 1) / NT;
    __shared__ T lds[2][TXH][ZH];

    const TileDev t = tiles[xcd_remap(blockIdx.x, ntiles)];
    const ShotDev<T>& S = shots[t.shot];
    const int nz = S.nz, nx = S.nx, nts = S.nts, wcap = S.wcap;
    const unsigned n = unsigned(nz) * unsigned(nx);
    const unsigned fbytes = n * SZ, colb = unsigned(nz) * SZ;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int iz = t.z0 + lane, zz = lane + FAT;
    const int c0 = FAT + w * R, ix0 = t.x0 + w * R;
    const unsigned voff = (unsigned(ix0) * unsigned(nz) + unsigned(iz)) * SZ;
    const bool zok = iz < nz - FAT;
    T cz[4], cx[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) cz[i] = S.cz[i], cx[i] = S.cx[i];
    const T dinv = S.filt[2 * S.h];  // 1/(2 dts)
    const unsigned hbase = (unsigned(t.x0 - FAT) * unsigned(nz) + unsigned(t.z0 - FAT)) * SZ;
    // halo fill: cells outside the update region are zero, as in k_imaging
    unsigned hv[NFILL];
#pragma unroll
    for (int it = 0; it < NFILL; ++it) {
        const int e = threadIdx.x + it * NT;
        const int c = e / ZH, z = e - c * ZH;
        const int hz = t.z0 - FAT + z, hx = t.x0 - FAT + c;
        const bool upd = e < TXH * ZH && hz >= FAT && hz < nz - FAT && hx >= FAT && hx < nx - FAT;
        hv[it] = upd ? hbase + unsigned(c) * colb + unsigned(z) * SZ : 0xfffffff0u;  // past the end: reads 0
    }
    auto slice = [&](const T* W, int j) { return make_rsrc(W + size_t(j % wcap) * n, fbytes); };
    const rsrc_t rdm = make_rsrc(S.dm, 5 * fbytes);
    T dm[5][R];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int f = 0; f < 5; ++f)
            dm[f][r] = zok && ix0 + r < nx - FAT ? bld<T>(rdm, voff, unsigned(r) * colb + unsigned(f) * fbytes) : T(0);

    const int step = ADJ ? -1 : 1;
    T fx[NFILL], fz[NFILL];   // the next sample's slice, in flight while this one is used
    auto prefetch = [&](int j) {
        const rsrc_t rwx = slice(S.Wvx, j), rwz = slice(S.Wvz, j);
#pragma unroll
        for (int it = 0; it < NFILL; ++it) {
            fx[it] = bld<T>(rwx, hv[it], 0u);
            fz[it] = bld<T>(rwz, hv[it], 0u);
        }
    };
    prefetch(j0);
    for (int j = j0;; j += step) {
        __syncthreads();
#pragma unroll
        for (int it = 0; it < NFILL; ++it) {
            const int e = threadIdx.x + it * NT;
            if (e < TXH * ZH) {
                (&lds[0][0][0])[e] = fx[it];
                (&lds[1][0][0])[e] = fz[it];
            }
        }
        __syncthreads();
        const bool more = j != j1;
        const rsrc_t rxm = slice(S.Wvx, j > 0 ? j - 1 : j), rzm = slice(S.Wvz, j > 0 ? j - 1 : j);
        const rsrc_t rxp = slice(S.Wvx, j < nts - 1 ? j + 1 : j), rzp = slice(S.Wvz, j < nts - 1 ? j + 1 : j);
        const rsrc_t rss = make_rsrc(S.ss[0] + size_t(j % S.sscap) * 5 * n, 5 * fbytes);
        T wxm[R], wzm[R], wxp[R], wzp[R], a[5][R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const unsigned so = unsigned(r) * colb;
            const bool ok = zok && ix0 + r < nx - FAT;
            wxm[r] = ok && j > 0 ? bld<T>(rxm, voff, so) : T(0);
            wzm[r] = ok && j > 0 ? bld<T>(rzm, voff, so) : T(0);
            wxp[r] = ok && j < nts - 1 ? bld<T>(rxp, voff, so) : T(0);
            wzp[r] = ok && j < nts - 1 ? bld<T>(rzp, voff, so) : T(0);
            if (ADJ) {
#pragma unroll
                for (int f = 0; f < 5; ++f) a[f][r] = ok ? bld<T>(rss, voff, so + unsigned(f) * fbytes) : T(0);
            }
        }
        if (more) prefetch(j + step);
        T xx[R], zxm[R];
        {
            T q[R + 8];
#pragma unroll
            for (int i = 0; i < R + 8; ++i) q[i] = lds[0][c0 - 4 + i][zz];
#pragma unroll
            for (int r = 0; r < R; ++r) xx[r] = dp_q(q, r + 4, cx);
#pragma unroll
            for (int i = 0; i < R + 8; ++i) q[i] = lds[1][c0 - 4 + i][zz];
#pragma unroll
            for (int r = 0; r < R; ++r) zxm[r] = dm_q(q, r + 4, cx);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const T zv = dp_q(&lds[1][c0 + r][zz], 0, cz);
            const T xz = dm_q(&lds[0][c0 + r][zz], 0, cz) + zxm[r];
            const T tx = j == 0 ? -wxp[r] : j == nts - 1 ? wxm[r] : wxm[r] - wxp[r];
            const T tz = j == 0 ? -wzp[r] : j == nts - 1 ? wzm[r] : wzm[r] - wzp[r];
            if (ADJ) {
                dm[0][r] = dm[0][r] + a[0][r] * tx * dinv;
                dm[1][r] = dm[1][r] + a[1][r] * tz * dinv;
                dm[2][r] = dm[2][r] + (a[2][r] + a[3][r]) * (xx[r] + zv);
                dm[3][r] = dm[3][r] + T(2) * (xx[r] * a[2][r] + zv * a[3][r]);
                dm[4][r] = dm[4][r] + a[4][r] * xz;
            } else if (zok && ix0 + r < nx - FAT) {
                const unsigned so = unsigned(r) * colb;
                const T dl = dm[2][r] * (xx[r] + zv);
                bst(rss, dm[0][r] * tx * dinv, voff, so);
                bst(rss, dm[1][r] * tz * dinv, voff, so + fbytes);
                bst(rss, dl + T(2) * dm[3][r] * xx[r], voff, so + 2 * fbytes);
                bst(rss, dl + T(2) * dm[3][r] * zv, voff, so + 3 * fbytes);
                bst(rss, dm[4][r] * xz, voff, so + 4 * fbytes);
            }
        }
        if (!more) break;
    }
    if (ADJ) {
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (zok && ix0 + r < nx - FAT) {
#pragma unroll
                for (int f = 0; f < 5; ++f) bst(rdm, dm[f][r], voff, unsigned(r) * colb + unsigned(f) * fbytes);
            }
    }
}

}  // namespace eio
