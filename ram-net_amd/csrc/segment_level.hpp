// Level-scheduled segment scan (gated sparse update + top-K read), top-K <= 16.
//
// Within a chunk of L = 32 tokens, an event (a slot write or read) only has to
// wait for the earlier writes of its own slot. Its level is the number of
// those writes in the chunk: the writes before its token for a write, the
// writes up to and including its token for a read (a token writes before it
// reads). Running
//     reads of level 0, writes of level 0, reads of level 1, writes of level 1, ...
// therefore reproduces the token order exactly, and almost every event has
// level 0 (88 % at 1024 slots and 8 events a token, 94 % at 4096 and 16). So
// a wave holds L tokens at once -- two lanes per token, VEC channels per lane
// -- and moves the rows of one event of all L tokens with one wide LDS
// instruction; the token-to-token chain of
// the one-token scan (segment_scan.hpp: one LDS round trip every four
// tokens, 180 cycles a token) becomes one round trip per level and chunk.
//
// Three parts:
//  * segment_schedule_kernel: per 32-token tile, every event's level, from a
//    per-slot bit mask of the tokens that write it (LDS atomic or; popcounts
//    of its lower bits are the levels). Each token's events are permuted so
//    that those of level >= 1 come first, which lets the scan bound the
//    later levels by a few event positions, counted per chunk and level.
//  * the mass wave of segment_level_kernel: the slot masses (one scalar per
//    slot), the same way, one chunk ahead; it stages each write's gain (and,
//    mass-aware, each read's effective weight) in LDS.
//  * the state waves: each owns CSW = VEC * LPT channels of the slice and an
//    LDS region of (A + 2) rows of them. LDS executes a wave's accesses in
//    program order, so the levels need no barrier. Progress counters in LDS
//    hand over the mass wave's stage, a ring of a few chunks, so the waves
//    drift apart and one's waits fall under another's work.
//
// Rows A and A + 1 of a region are dummies: an event outside the level at
// hand reads row A (zeros) and writes row A + 1 (never read). An event word
// is level << 24 | slot, so subtracting level << 24 and taking the unsigned
// minimum with the dummy row selects both at once.
#pragma once

#include "ramnet_device.hpp"
#include "ramnet_kernels.hpp"
#include "segment_scan.hpp"

namespace ramnet {

constexpr int kTile = 32;                 // tokens per chunk, and per tile of the schedule arrays (kScanPad)
constexpr uint32_t kNoEvent = 0xff000000u;  // level 255: an event that never acts
constexpr int kLevelMaxWaves = 4;         // state waves of a workgroup
constexpr int kLevelRing = 4;             // chunks of gains the mass wave may be ahead

// Schedule arrays, in the part of the workspace that holds the gain records
// and flags of the other forms (16 bytes per event of the larger top-K and 4
// per token): per 32-token tile, event-major rows of 32 tokens.
//   write   Kw words  level << 24 | slot, events in scan order
//   mass    Kw words  level << 24 | position << 16 | slot, events in decoder order
//   read    Kr pairs  {level << 24 | slot, read weight}, in scan order
//   counts  per chunk, word 0: its late levels n (bits 0..7), and the event
//           positions holding a read of level L (bits 8..15); word l = 1 ..
//           n: the positions holding a read (bits 0..7) and a write (bits
//           8..15) of level l < L. Bit 31 of the call's first word: another
//           form takes the call (crowd_kernel)
struct LevelSchedule {
    uint32_t *write, *mass;
    uint2 *read;
    uint32_t *counts;
};
// (of head bh)
__host__ __device__ inline LevelSchedule level_schedule(const SegmentJob &job, int t_pad, int bh) {
    LevelSchedule s;
    s.write = reinterpret_cast<uint32_t *>(job.gain + static_cast<int64_t>(bh) * t_pad * (job.Kw > job.Kr ? job.Kw : job.Kr));
    s.mass = s.write + static_cast<int64_t>(t_pad) * job.Kw;
    s.read = reinterpret_cast<uint2 *>(s.mass + static_cast<int64_t>(t_pad) * job.Kw);
    s.counts = reinterpret_cast<uint32_t *>(job.flags) + static_cast<int64_t>(bh) * t_pad;
    return s;
}

struct LevelGeom {
    int n_units;   // B * H * n_slices
    int n_slices;  // ceil(C / (nw * CSW))
    int t_pad;
    int nw;        // state waves (1, 2 or 4)
    CrowdRule crowd;  // set: a crowded call is left to another form
};

// LDS of a workgroup: the state regions, the masses, the stage ring and the
// progress counters.
inline size_t level_lds_bytes(int A, int vec, int nw, int km, bool ma) {
    return (static_cast<size_t>(A + 2) * (2 * vec * nw + 1) * 4 + 15) / 16 * 16 +
           static_cast<size_t>(kLevelRing) * kTile * (km + 4) * 4 * (ma ? 2 : 1) + (kLevelMaxWaves + 1) * 4;
}
// LDS of the schedule kernel: a 32-bit token mask per slot for each of the
// two tiles of a wave.
inline size_t schedule_lds_bytes(int A) { return static_cast<size_t>(A) * 2 * 4; }

// One wave per 64 tokens (two tiles) of one (b, h), one token per lane.
// Bound by its record traffic (24 bytes per write and 16 per read).
template<int KM>
__global__ __launch_bounds__(kWave) void segment_schedule_kernel(const SegmentJob job, int t_pad) {
    constexpr int L = kTile;
    extern __shared__ __align__(16) uint32_t masks[];
    __shared__ int late[4][L + 1];  // per tile: positions holding a read, a write of each level
    const int A = job.A, Kw = job.Kw, Kr = job.Kr;
    const int per_head = (t_pad + kWave - 1) / kWave;
    const int bh = static_cast<int>(blockIdx.x) / per_head;
    const int lane = static_cast<int>(threadIdx.x);
    const int t = (static_cast<int>(blockIdx.x) - bh * per_head) * kWave + lane;
    const bool in = t < t_pad;
    const int tc = in ? t : t_pad - 1;
    for (int i = lane; i < 2 * A; i += kWave)
        masks[i] = 0;
    for (int i = lane; i < 4 * (L + 1); i += kWave)
        (&late[0][0])[i] = 0;
    // (every load issued up front, from clamped event indices)
    const WriteRec *gw = job.wrec + static_cast<int64_t>(bh) * Kw * t_pad + tc;
    const ReadRec *gr = job.rrec + static_cast<int64_t>(bh) * Kr * t_pad + tc;
    int ws[KM], rs[KM];
    float rr[KM];
#pragma unroll
    for (int k = 0; k < KM; ++k) {
        ws[k] = gw[static_cast<uint32_t>(min(k, Kw - 1) * t_pad)].slot;
        const int2 q = *reinterpret_cast<const int2 *>(gr + static_cast<uint32_t>(min(k, Kr - 1) * t_pad));
        rs[k] = q.x;
        rr[k] = __int_as_float(q.y);
    }
#pragma unroll
    for (int k = 0; k < KM; ++k) {
        ws[k] = (in & (k < Kw)) ? ws[k] : -2;
        rs[k] = (in & (k < Kr)) ? rs[k] : -1;
    }
    const int tt = lane % kTile;
    uint32_t *mine = masks + (lane / kTile) * A;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KM; ++k)
        if (ws[k] >= 0)
            atomicOr(&mine[ws[k]], 1u << tt);
    __syncthreads();
    // bits of the tokens of this token's chunk before it, and up to it
    const uint32_t before = (1u << tt) - 1, upto = (2u << tt) - 1;
    uint32_t wl[KM], rl[KM];  // levels; 255 for events that do not act
    int wx = 0, rx = 0;       // this token's events of level >= 1
#pragma unroll
    for (int k = 0; k < KM; ++k) {
        const uint32_t mw = mine[max(ws[k], 0)], mr = mine[max(rs[k], 0)];
        wl[k] = ws[k] >= 0 ? __popc(mw & before) : 255u;
        rl[k] = rs[k] >= 0 ? __popc(mr & upto) : 255u;
        wx += (wl[k] != 0) & (wl[k] != 255u);
        rx += (rl[k] != 0) & (rl[k] != 255u);
    }
    const LevelSchedule out = level_schedule(job, t_pad, bh);
    const int tile = tc / kTile;
    uint32_t *ow = out.write + tile * Kw * kTile + tt, *om = out.mass + tile * Kw * kTile + tt;
    uint2 *orw = out.read + tile * Kr * kTile + tt;
    int wp[KM], rp[KM];  // positions in scan order
    int wlate = 0, rlate = 0, wzero = wx, rzero = rx;
#pragma unroll
    for (int k = 0; k < KM; ++k) {
        const bool we = (wl[k] != 0) & (wl[k] != 255u), re = (rl[k] != 0) & (rl[k] != 255u);
        wp[k] = we ? wlate : wzero;
        rp[k] = re ? rlate : rzero;
        wlate += we;
        wzero += !we;
        rlate += re;
        rzero += !re;
    }
    if (in) {
#pragma unroll
        for (int k = 0; k < KM; ++k) {
            if (k < Kw) {
                const uint32_t s = static_cast<uint32_t>(max(ws[k], 0));
                ow[wp[k] * kTile] = wl[k] << 24 | s;
                om[k * kTile] = wl[k] << 24 | static_cast<uint32_t>(wp[k]) << 16 | s;
            }
            if (k < Kr) {
                orw[rp[k] * kTile] =
                    make_uint2(rl[k] << 24 | static_cast<uint32_t>(max(rs[k], 0)), __float_as_uint(rr[k]));
            }
        }
    }
    // positions per level of each chunk, and its levels (contiguous from 1: an
    // event of a level waits for one of each level below). Through LDS
    // maxima: 34 us for 128 heads, T = 4096, K = 8, spread or crowded; a
    // butterfly over the lanes per level took 35 us on spread addresses and
    // 61 on crowded ones, whose chunks have up to 32 levels.
    const int half = lane / kTile * 2;
#pragma unroll
    for (int k = 0; k < KM; ++k) {
        if ((rl[k] != 0) & (rl[k] != 255u))
            atomicMax(&late[half][rl[k]], rp[k] + 1);
        if ((wl[k] != 0) & (wl[k] != 255u))
            atomicMax(&late[half + 1][wl[k]], wp[k] + 1);
    }
    __syncthreads();
    // lane l of a tile: level l, and level L in word 0
    const uint32_t n = late[half][tt] | late[half + 1][tt] << 8, last = late[half][L];
    const uint32_t any = static_cast<uint32_t>(__ballot((tt > 0) & (n != 0)) >> (lane / kTile * kTile));
    const uint32_t levels = last != 0 ? L | last << 8 : any != 0 ? 31 - __clz(static_cast<int>(any)) : 0;
    if (in)
        out.counts[tc] = tt == 0 ? levels : n;
}

// Orders LDS accesses of different lanes for the compiler (the hardware runs
// a wave's accesses in program order).
__device__ __forceinline__ void lds_phase() { asm volatile("" ::: "memory"); }
// VEC activation elements through a buffer resource (voff: bytes of this
// lane, soff: uniform bytes); loads past the resource return 0, stores past
// it are dropped.
template<typename Scalar, int VEC>
__device__ __forceinline__ XBits<Scalar, VEC> buffer_x(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    XBits<Scalar, VEC> x;
    constexpr int B = VEC * static_cast<int>(sizeof(Scalar));
    if constexpr (B == 2) {
        x.w[0] = __builtin_amdgcn_raw_buffer_load_b16(r, voff, soff, 0);
    } else if constexpr (B == 4) {
        x.w[0] = __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0);
    } else if constexpr (B == 8) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0);
        x.w[0] = v[0];
        x.w[1] = v[1];
    } else {
        static_assert(B == 16, "2 to 16 bytes");
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
        x.w[0] = v[0];
        x.w[1] = v[1];
        x.w[2] = v[2];
        x.w[3] = v[3];
    }
    return x;
}
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template<typename Scalar, int VEC>
__device__ __forceinline__ void buffer_y(__amdgpu_buffer_rsrc_t r, int voff, int soff, const FVec<VEC> &v) {
    if constexpr (sizeof(Scalar) == 4) {
        if constexpr (VEC == 1)
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v.v[0]), r, voff, soff, 0);
        else if constexpr (VEC == 2)
            __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(v.v[0]), __float_as_uint(v.v[1])}, r, voff, soff, 0);
        else
            __builtin_amdgcn_raw_buffer_store_b128(u32x4{__float_as_uint(v.v[0]), __float_as_uint(v.v[1]),
                                                         __float_as_uint(v.v[2]), __float_as_uint(v.v[3])}, r, voff, soff, 0);
    } else {
        uint32_t w[(VEC + 1) / 2];
#pragma unroll
        for (int i = 0; i < (VEC + 1) / 2; ++i)
            w[i] = to_bits16<Scalar>(v.v[2 * i]) |
                   (2 * i + 1 < VEC ? static_cast<uint32_t>(to_bits16<Scalar>(v.v[2 * i + 1 < VEC ? 2 * i + 1 : 0])) << 16 : 0u);
        if constexpr (VEC == 1)
            __builtin_amdgcn_raw_buffer_store_b16(static_cast<uint16_t>(w[0]), r, voff, soff, 0);
        else if constexpr (VEC == 2)
            __builtin_amdgcn_raw_buffer_store_b32(w[0], r, voff, soff, 0);
        else
            __builtin_amdgcn_raw_buffer_store_b64(u32x2{w[0], w[1]}, r, voff, soff, 0);
    }
}

// MODE 0: any shape. 1: every lane owns VEC real channels, its x and y
// elements are aligned for one wide access and a head's x and y lie within
// 2^31 bytes. 2: also Kw == Kr == KM.
template<typename Scalar, int KM, int VEC, bool MA, int MODE>
__global__ __launch_bounds__(kWave *(kLevelMaxWaves + 1)) void segment_level_kernel(const SegmentJob job,
                                                                                    const LevelGeom geo) {
    constexpr bool FULL = MODE >= 1, EXACT = MODE == 2;
    constexpr int LPT = 2;  // lanes per token
    constexpr int L = kTile;
    constexpr int CSW = VEC * LPT;
    constexpr int KQ = KM / LPT;  // mass wave: events per lane of a token
    static_assert(KM % LPT == 0 && L * LPT == kWave, "lane layout");
    extern __shared__ __align__(16) float lds[];
    const int NW = geo.nw;
    const int CS = NW * CSW;
    // each XCD gets a contiguous run of units: the slices of a head share an L2
    const int per_xcd = (geo.n_units + 7) / 8;
    const int unit = static_cast<int>(blockIdx.x % 8) * per_xcd + static_cast<int>(blockIdx.x / 8);
    if (unit >= geo.n_units)
        return;
    const int tid = static_cast<int>(threadIdx.x), nthreads = kWave * (NW + 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int lane = tid % kWave;
    const int bh = unit / geo.n_slices;
    const int c0 = (unit - bh * geo.n_slices) * CS;
    const int A = job.A, C = job.C, T = job.T, Kw = job.Kw, Kr = job.Kr, Tp = geo.t_pad;
    if (geo.crowd.flags && crowded(geo.crowd))
        return;
    const int rs = (A + 2) * CSW;  // floats per wave region
    constexpr int SV = CSW % 4 == 0 ? 4 : 2;  // floats per state access
    auto region = [&](int c) { return lds + c / CSW * rs + c % CSW; };  // slice channel c in slot 0
    float *ms = lds + static_cast<size_t>(rs) * NW;
    // stage: [chunk % ring][token][position] gains and, mass-aware, effective read weights
    constexpr int SR = KM + 4;  // floats per token (16-byte rows off the bank period)
    constexpr int NB = kLevelRing;
    float *stage = lds + (static_cast<size_t>(A + 2) * (CS + 1) + 3) / 4 * 4;
    float *stage_r = stage + NB * L * SR;
    // progress: chunks finished by each state wave, then chunks staged by the mass wave
    using LdsCounter = volatile __attribute__((address_space(3))) int *;
    const LdsCounter finished = (LdsCounter)(uintptr_t)lds_addr(stage + NB * L * SR * (MA ? 2 : 1));
    const LdsCounter staged = finished + kLevelMaxWaves;
    auto post = [&](LdsCounter p, int v) {
        lds_phase();
        if (lane == 0)
            *p = v;
    };

    // ---- state slice and masses -> LDS
    {
        const float *src = job.init_slot + static_cast<int64_t>(bh) * A * C + c0;
        if (FULL && (C & (SV - 1)) == 0 && (reinterpret_cast<uintptr_t>(job.init_slot) & (4 * SV - 1)) == 0) {
            // rows of the slice in SV-float pieces, eight loads in flight per thread
            const int lq = __builtin_ctz(static_cast<unsigned>(CS / SV)), n = A << lq;
            for (int i0 = tid; i0 < n; i0 += 8 * nthreads) {
                FVec<SV> v[8];
                float *to[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int i = min(i0 + j * nthreads, n - 1);
                    const int a = i >> lq, c = (i & ((1 << lq) - 1)) * SV;
                    to[j] = region(c) + a * CSW;
                    v[j] = lds_load<SV>(src + static_cast<int64_t>(a) * C + c);
                }
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    lds_store<SV>(to[j], v[j]);
            }
        } else {
            for (int i = tid; i < A * CS; i += nthreads) {
                const int a = i / CS, c = i - a * CS;
                const bool ok = c0 + c < C;
                const float v = src[static_cast<int64_t>(a) * C + (ok ? c : 0)];
                region(c)[a * CSW] = ok ? v : 0.f;
            }
        }
        for (int i = tid; i < 2 * CS; i += nthreads)
            lds[(i / (2 * CSW)) * rs + A * CSW + i % (2 * CSW)] = 0.f;
        const float *msrc = job.init_mass + static_cast<int64_t>(bh) * A;
        for (int a = tid; a < A + 2; a += nthreads)
            ms[a] = a < A ? msrc[a] : 1.f;
        for (int i = tid; i < NB * L * SR * (MA ? 2 : 1) + kLevelMaxWaves + 1; i += nthreads)
            stage[i] = 0.f;
    }
    const LevelSchedule sch = level_schedule(job, Tp, bh);
    // one resource per array over this head's part; loads take a constant
    // byte offset per lane and a scalar one per chunk and event, so they cost
    // no vector address arithmetic
    auto head_rsrc = [&](const void *base, int K) {
        const int bytes = Tp * K * 4;
        return __builtin_amdgcn_make_buffer_rsrc(
            const_cast<void *>(base), 0, bytes, kBufWord3);
    };
    const auto b_write = head_rsrc(sch.write, Kw), b_mass = head_rsrc(sch.mass, Kw);
    const auto b_read = head_rsrc(sch.read, 2 * Kr);
    const auto b_counts = head_rsrc(sch.counts, 1);
    // byte offset of chunk c in an array of K words per token
    auto chunk_off = [&](int c, int K) { return c * K * kTile * 4; };
    const int tl = lane / LPT, sub = lane % LPT;  // token of the chunk; lane of the token
    const int nc = (T + L - 1) / L;
    const int cnt_off = min(lane, L - 1) * 4;
    auto chunk_at = [&](int c) { return min(c, nc - 1); };
    __syncthreads();

    if (wave == NW) {
        // ---- mass wave
        // the lane's events: sub + LPT * i, in decoder order (writes) and scan order (reads)
        bool onw[KQ], onr[KQ];
        int vw[KQ], vr[KQ], vrec[KQ];
#pragma unroll
        for (int i = 0; i < KQ; ++i) {
            const int k = sub + LPT * i;
            onw[i] = k < Kw;
            onr[i] = k < Kr;
            vw[i] = (min(k, Kw - 1) * kTile + tl) * 4;
            vr[i] = (min(k, Kr - 1) * kTile + tl) * 8;
            vrec[i] = (min(k, Kw - 1) * Tp + tl) * static_cast<int>(sizeof(WriteRec)) + 4;  // at w, alpha
        }
        const auto b_rec = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<WriteRec *>(job.wrec) + static_cast<int64_t>(bh) * Kw * Tp, 0,
            Kw * Tp * static_cast<int>(sizeof(WriteRec)), kBufWord3);
        struct Fetch {
            uint32_t word[KQ], rword[KQ];
            float w[KQ], al[KQ], r[KQ];
            uint32_t cnt;
        };
        auto fetch = [&](int c, Fetch &f) {
            const int ow = chunk_off(c, Kw), orr = 2 * chunk_off(c, Kr);
#pragma unroll
            for (int i = 0; i < KQ; ++i) {
                f.word[i] = __builtin_amdgcn_raw_buffer_load_b32(b_mass, vw[i], ow, 0);
                // (w and alpha alone: the unused parts of a 16-byte load would
                // be reused as temporaries, which waits for the load)
                const auto q = __builtin_amdgcn_raw_buffer_load_b64(b_rec, vrec[i], c * L * static_cast<int>(sizeof(WriteRec)), 0);
                f.w[i] = __uint_as_float(q[0]);
                f.al[i] = __uint_as_float(q[1]);
                if constexpr (MA) {
                    const auto rd = __builtin_amdgcn_raw_buffer_load_b64(b_read, vr[i], orr, 0);
                    f.rword[i] = rd[0];
                    f.r[i] = __uint_as_float(rd[1]);
                }
            }
            f.cnt = __builtin_amdgcn_raw_buffer_load_b32(b_counts, cnt_off, c * L * 4, 0);
        };
        const float eps = job.eps;
        auto run = [&](const Fetch &f, int buf) {
            float g[KQ], mr[KQ];
            uint32_t word[KQ], rword[KQ];
#pragma unroll
            for (int i = 0; i < KQ; ++i) {
                g[i] = 0.f;
                mr[i] = 0.f;
                word[i] = EXACT || onw[i] ? f.word[i] : kNoEvent;
                if constexpr (MA)
                    rword[i] = EXACT || onr[i] ? f.rword[i] : kNoEvent;
            }
            auto level = [&](uint32_t l) {
                const uint32_t off = l << 24;
                if constexpr (MA) {
#pragma unroll
                    for (int i = 0; i < KQ; ++i) {
                        const uint32_t s = rword[i] - off;
                        const float m = ms[min(s, static_cast<uint32_t>(A))];
                        mr[i] = s < 0x1000000u ? m : mr[i];
                    }
                }
                float m[KQ];
                uint32_t at[KQ];
                bool hit[KQ];
#pragma unroll
                for (int i = 0; i < KQ; ++i) {
                    const uint32_t s = word[i] - off;
                    hit[i] = s < 0x1000000u;
                    at[i] = hit[i] ? s & 0xffffu : static_cast<uint32_t>(A) + 1;
                    m[i] = ms[at[i]];
                }
#pragma unroll
                for (int i = 0; i < KQ; ++i) {
                    const float m2 = fmaf(f.al[i], m[i], f.w[i]);
                    ms[at[i]] = m2;
                    g[i] = hit[i] ? scan_gain(f.w[i], m2 + eps) : g[i];
                }
                lds_phase();
            };
            const int n = readlane_i(static_cast<int>(f.cnt), 0) & 0xff;
#pragma unroll 1
            for (int l = 0; l <= n; ++l)
                level(l);
            float *sg = stage + (buf * L + tl) * SR;
#pragma unroll
            for (int i = 0; i < KQ; ++i)
                if (EXACT || onw[i])
                    sg[(f.word[i] >> 16) & 0xffu] = g[i];
            if constexpr (MA) {
                float sr = 0.f, srm = 0.f, wm[KQ];
#pragma unroll
                for (int i = 0; i < KQ; ++i) {
                    const float r = onr[i] ? f.r[i] : 0.f;
                    wm[i] = r * mr[i];
                    sr += r;
                    srm += wm[i];
                }
                const float scale = event_sum<LPT>(sr) / (event_sum<LPT>(srm) + eps);
                float *sw = stage_r + (buf * L + tl) * SR;
#pragma unroll
                for (int i = 0; i < KQ; ++i)
                    if (onr[i])
                        sw[sub + LPT * i] = wm[i] * scale;
            }
        };
        // Chunk c goes to ring slot c % NB once every state wave has finished
        // chunk c - NB. A wave that sees a counter also sees what was stored
        // before it (each wave's LDS accesses execute in order).
        int freed = 0;
        auto produce = [&](const Fetch &f, int c) {
            while (freed < c - NB + 1) {
                const int m = finished[min(lane, NW - 1)];
                freed = readlane_i(m, 0);
#pragma unroll
                for (int w = 1; w < kLevelMaxWaves; ++w)
                    freed = min(freed, readlane_i(m, w));
                if (freed < c - NB + 1)
                    __builtin_amdgcn_s_sleep(1);
            }
            run(f, c & (NB - 1));
            post(staged, c + 1);
        };
        Fetch fa, fb;
        fetch(0, fa);
        for (int c = 0; c < nc; c += 2) {
            fetch(chunk_at(c + 1), fb);
            __builtin_amdgcn_sched_barrier(0);
            produce(fa, c);
            if (c + 1 >= nc)
                break;
            fetch(chunk_at(c + 2), fa);
            __builtin_amdgcn_sched_barrier(0);
            produce(fb, c + 1);
        }
        if (c0 == 0) {
            float *mdst = job.mass_out + static_cast<int64_t>(bh) * A;
            for (int a = lane; a < A; a += kWave)
                mdst[a] = ms[a];
        }
    } else {
        // ---- state waves
        const int ch = c0 + wave * CSW + sub * VEC;  // first channel of this lane
        const int b = bh / job.H, h = bh - b * job.H;
        const Scalar *gx = static_cast<const Scalar *>(job.x) + b * job.x_stride[0] + h * job.x_stride[1];
        Scalar *gy = static_cast<Scalar *>(job.y) + b * job.y_stride[0] + h * job.y_stride[1];
        const int64_t xt = job.x_stride[2], yt = job.y_stride[2];
        const uint32_t base = lds_addr(lds + static_cast<size_t>(wave) * rs) + static_cast<uint32_t>(sub * VEC * 4);
        const uint32_t zero_row = static_cast<uint32_t>(A), trash_row = zero_row + 1;
        constexpr int ES = static_cast<int>(sizeof(Scalar));
        // FULL: x and y of this head through resources that end at its last
        // token (loads past T give 0, stores past T are dropped)
        const auto b_x = __builtin_amdgcn_make_buffer_rsrc(const_cast<Scalar *>(gx), 0,
                                                           FULL ? static_cast<int>(((T - 1) * xt + C) * ES) : 0, kBufWord3);
        const auto b_y = __builtin_amdgcn_make_buffer_rsrc(gy, 0, FULL ? static_cast<int>(((T - 1) * yt + C) * ES) : 0,
                                                           kBufWord3);
        const int vx = static_cast<int>(tl * xt + ch) * ES, vy = static_cast<int>(tl * yt + ch) * ES;
        const int sx = static_cast<int>(xt) * L * ES, sy = static_cast<int>(yt) * L * ES;  // bytes per chunk
        const int vt = tl * 4;
        struct Fetch {
            uint32_t w[KM], r[KM], wt[MA ? 1 : KM];
            XBits<Scalar, VEC> x;
            uint32_t cnt;
        };
        auto fetch = [&](int c, Fetch &f) {
            const int ow = chunk_off(c, Kw), orr = 2 * chunk_off(c, Kr);
#pragma unroll
            for (int k = 0; k < KM; ++k) {
                // (rows past an array's top-K hold other events or lie past
                // the resource; they are masked below)
                if constexpr (MA) {
                    f.r[k] = __builtin_amdgcn_raw_buffer_load_b32(b_read, 2 * (vt + k * kTile * 4), orr, 0);
                } else {
                    const auto rd = __builtin_amdgcn_raw_buffer_load_b64(b_read, 2 * (vt + k * kTile * 4), orr, 0);
                    f.r[k] = rd[0];
                    f.wt[k] = rd[1];
                }
                f.w[k] = __builtin_amdgcn_raw_buffer_load_b32(b_write, vt + k * kTile * 4, ow, 0);
            }
            if constexpr (FULL)
                f.x = buffer_x<Scalar, VEC>(b_x, vx, c * sx);
            else
                f.x = load_x_bits<Scalar, VEC, false>(gx + min(c * L + tl, T - 1) * xt, ch, C);
            f.cnt = __builtin_amdgcn_raw_buffer_load_b32(b_counts, cnt_off, c * L * 4, 0);
        };
        auto row = [&](uint32_t word, uint32_t off, uint32_t dummy) {
            return lds_at(base + min(word - off, dummy) * static_cast<uint32_t>(CSW * 4));
        };
        int seen = 0;  // chunks staged, when last looked at
        auto run = [&](const Fetch &f, int c) {
            uint32_t ww[KM], rw[KM];
            float wt[KM], g[KM];
            FVec<VEC> s[KM], r[KM];
            float *p[KM], *q[KM];
            while (seen <= c)
                seen = __builtin_amdgcn_readfirstlane(*staged);
            lds_phase();
            const float *sg = stage + ((c & (NB - 1)) * L + tl) * SR, *sw = stage_r + ((c & (NB - 1)) * L + tl) * SR;
#pragma unroll
            for (int i = 0; i < KM / 4; ++i) {
                const FVec<4> g4 = lds_load<4>(sg + 4 * i);
                FVec<4> w4;
                if constexpr (MA)
                    w4 = lds_load<4>(sw + 4 * i);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    g[4 * i + v] = g4.v[v];
                    if constexpr (MA)
                        wt[4 * i + v] = w4.v[v];
                }
            }
            // events past the top-K (uniform) never act
#pragma unroll
            for (int k = 0; k < KM; ++k) {
                ww[k] = f.w[k] | (EXACT || k < Kw ? 0u : kNoEvent);
                rw[k] = f.r[k] | (EXACT || k < Kr ? 0u : kNoEvent);
                if constexpr (!MA)
                    wt[k] = __uint_as_float(EXACT || k < Kr ? f.wt[k] : 0u);
                q[k] = row(rw[k], 0, zero_row);
                p[k] = row(ww[k], 0, trash_row);
            }
#pragma unroll
            for (int k = 0; k < KM; ++k)
                r[k] = lds_load<VEC>(q[k]);
#pragma unroll
            for (int k = 0; k < KM; ++k)
                s[k] = lds_load<VEC>(p[k]);
            __builtin_amdgcn_sched_barrier(0);
            const FVec<VEC> x = x_bits_to_f<Scalar, VEC>(f.x);
            FVec<VEC> acc;
#pragma unroll
            for (int v = 0; v < VEC; ++v)
                acc.v[v] = 0.f;
            auto add = [&](int k) {
#pragma unroll
                for (int v = 0; v < VEC; ++v)
                    acc.v[v] = fmaf(wt[k], r[k].v[v], acc.v[v]);
            };
            auto update = [&](int k) {
#pragma unroll
                for (int v = 0; v < VEC; ++v)
                    s[k].v[v] = fmaf(g[k], x.v[v] - s[k].v[v], s[k].v[v]);
                lds_store<VEC>(p[k], s[k]);
            };
#pragma unroll
            for (int k = 0; k < KM; ++k)
                add(k);
#pragma unroll
            for (int k = 0; k < KM; ++k)
                update(k);
            lds_phase();
            // later levels: the first few positions, four at a time (two where
            // no more are needed); the first reads and writes load together
            const int head = readlane_i(static_cast<int>(f.cnt), 0), levels = head & 0xff;
#pragma unroll 1
            for (int l = 1; l <= levels; ++l) {
                const int n = l < L ? readlane_i(static_cast<int>(f.cnt), l) : head >> 8;
                const int nr = n & 0xff, nw = n >> 8;
                const uint32_t off = static_cast<uint32_t>(l) << 24;
                auto load_r = [&](int k) { r[k] = lds_load<VEC>(row(rw[k], off, zero_row)); };
                auto load_w = [&](int k) {
                    p[k] = row(ww[k], off, trash_row);
                    s[k] = lds_load<VEC>(p[k]);
                };
                load_r(0);
                load_r(1);
                if (nr > 2) {
                    load_r(2);
                    load_r(3);
                }
                load_w(0);
                load_w(1);
                if (nw > 2) {
                    load_w(2);
                    load_w(3);
                }
                add(0);
                add(1);
                if (nr > 2) {
                    add(2);
                    add(3);
#pragma unroll
                    for (int k0 = 4; k0 < KM; k0 += 4) {
                        if (nr > k0) {
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                load_r(k0 + j);
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                add(k0 + j);
                        }
                    }
                }
                lds_phase();
                update(0);
                update(1);
                if (nw > 2) {
                    update(2);
                    update(3);
#pragma unroll
                    for (int k0 = 4; k0 < KM; k0 += 4) {
                        if (nw > k0) {
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                load_w(k0 + j);
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                update(k0 + j);
                        }
                    }
                }
                lds_phase();
            }
            if constexpr (FULL) {
                buffer_y<Scalar, VEC>(b_y, vy, c * sy, acc);
            } else {
                const int t = c * L + tl;
                if (t < T) {
                    Scalar *yp = gy + t * yt + ch;
#pragma unroll
                    for (int v = 0; v < VEC; ++v)
                        if (ch + v < C)
                            store_out(yp + v, acc.v[v]);
                }
            }
            post(finished + wave, c + 1);
        };
        Fetch fa, fb;
        fetch(0, fa);
        for (int c = 0; c < nc; c += 2) {
            fetch(chunk_at(c + 1), fb);
            __builtin_amdgcn_sched_barrier(0);
            run(fa, c);
            if (c + 1 >= nc)
                break;
            fetch(chunk_at(c + 2), fa);
            __builtin_amdgcn_sched_barrier(0);
            run(fb, c + 1);
        }
    }
    __syncthreads();
    // ---- LDS -> post state
    {
        float *dst = job.slot_out + static_cast<int64_t>(bh) * A * C + c0;
        if (FULL && (C & (SV - 1)) == 0 && (reinterpret_cast<uintptr_t>(job.slot_out) & (4 * SV - 1)) == 0) {
            const int lq = __builtin_ctz(static_cast<unsigned>(CS / SV)), n = A << lq;
            for (int i0 = tid; i0 < n; i0 += 8 * nthreads) {
                FVec<SV> v[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int i = min(i0 + j * nthreads, n - 1);
                    v[j] = lds_load<SV>(region((i & ((1 << lq) - 1)) * SV) + (i >> lq) * CSW);
                }
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int i = min(i0 + j * nthreads, n - 1);
                    lds_store<SV>(dst + static_cast<int64_t>(i >> lq) * C + (i & ((1 << lq) - 1)) * SV, v[j]);
                }
            }
        } else {
            for (int i = tid; i < A * CS; i += nthreads) {
                const int a = i / CS, c = i - a * CS;
                if (c0 + c < C)
                    dst[static_cast<int64_t>(a) * C + c] = region(c)[a * CSW];
            }
        }
    }
}

template<typename Scalar, int KM, int VEC>
hipError_t launch_level(const SegmentJob &job, const LevelGeom &geo, bool full, hipStream_t stream) {
    const unsigned blocks = static_cast<unsigned>(((geo.n_units + 7) / 8) * 8);
    const dim3 threads(kWave * (geo.nw + 1));
    const size_t lds = level_lds_bytes(job.A, VEC, geo.nw, KM, job.mass_aware != 0);
    const int mode = !full ? 0 : job.Kw == KM && job.Kr == KM ? 2 : 1;
#define RAMNET_LEVEL(MA, MODE)                                                                                        \
    if ((job.mass_aware != 0) == MA && mode == MODE)                                                                  \
        hipLaunchKernelGGL((segment_level_kernel<Scalar, KM, VEC, MA, MODE>), dim3(blocks), threads, lds, stream, job, \
                           geo)
    RAMNET_LEVEL(false, 0);
    RAMNET_LEVEL(false, 1);
    RAMNET_LEVEL(false, 2);
    RAMNET_LEVEL(true, 0);
    RAMNET_LEVEL(true, 1);
    RAMNET_LEVEL(true, 2);
#undef RAMNET_LEVEL
    return hipGetLastError();
}

// Channels per lane compiled: 4, 2 or 1; with 16 events 2 or 1 (4 would hold
// 16 rows of 4 channels twice and spill).
constexpr bool level_layout_compiled(int km, int vec) { return vec == 1 || vec == 2 || (vec == 4 && km <= 8); }

template<typename Scalar>
hipError_t level_dispatch(const SegmentJob &job, const LevelGeom &geo, int vec, int km, bool full, hipStream_t stream) {
#define RAMNET_LEVEL_CASE(K, V) \
    if (km == K && vec == V) return launch_level<Scalar, K, V>(job, geo, full, stream);
    RAMNET_LEVEL_CASE(4, 4)
    RAMNET_LEVEL_CASE(4, 2)
    RAMNET_LEVEL_CASE(4, 1)
    RAMNET_LEVEL_CASE(8, 4)
    RAMNET_LEVEL_CASE(8, 2)
    RAMNET_LEVEL_CASE(8, 1)
    RAMNET_LEVEL_CASE(16, 2)
    RAMNET_LEVEL_CASE(16, 1)
#undef RAMNET_LEVEL_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_level_f32(const SegmentJob &, const LevelGeom &, int, int, bool, hipStream_t);
hipError_t launch_level_f16(const SegmentJob &, const LevelGeom &, int, int, bool, hipStream_t);
hipError_t launch_level_bf16(const SegmentJob &, const LevelGeom &, int, int, bool, hipStream_t);

}  // namespace ramnet
