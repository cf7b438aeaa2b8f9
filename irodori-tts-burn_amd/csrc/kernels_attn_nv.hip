// Flash attention on 16-bit operands as a caller has them: Q, K, V [B, H, S, Dh] row-major
// (Dh 64 or 128), a float key mask, no staging pass (irodori_op_sdpa / _noalloc and the
// condition encoders; fused_sdpa_native.rs:220-302, attention.rs:52-127 semantics).
//
// Per 64-key tile and wavefront (32 queries), on the 32x32x16 matrix-core shape:
//   S^T = K Q^T      K tile from LDS (A operand), Q^T in registers (B operand): lane l holds
//                    query l % 32 and keys 8a + 4 (l / 32) + c of every 16-key group.
//   softmax          in f32: p = exp2(s c - m) with c = scale log2(e), one FMA and one
//                    exponential an element.  The reference m is lazy: a query's first tile with
//                    a score above -inf sets it, and it moves when a lane's sum of p over a tile
//                    shows a p that may exceed the slack.
//   O^T += V^T P^T   P^T is the S^T accumulator; the matching V^T operand (4 consecutive keys
//                    of one dim per lane, twice) comes out of the row-major V tile by
//                    ds_read_b64_tr_b16, the transposing LDS read, so V needs no transposed
//                    copy in memory.
// Workgroup: QB query blocks x KVS key parities; tiles are dealt to the parities round-robin
// and the partial (m, l, O) merged through LDS.  K and V tiles move HBM -> LDS with
// buffer_load_dwordx4 ... lds (rows past the last key read as zero).
//
// What bounds it: with about one wavefront per SIMD, a tile step's chain of barrier, LDS reads,
// 32 quarter-rate exponentials and ~90 other VALU operations, and the P V MFMAs.  At the
// published model's call (1 x 20 heads, 750 queries, 950 keys of which 80 % valid, 64-dim): 12.1
// us back to back, where staging Q, V^T and the key bits in a buffer allocated per call took 8.0
// us before a 9.9 us attention (30 us a call with the allocation and the gap); 1 x 10 x 256 x 256
// at 128-dim 9.5 against 21.8 us on 16x16 tiles with one 16-query block per wavefront.
#include <type_traits>

#include "attn_util.hpp"
#include "kernels.hpp"

namespace irodori {

namespace {

constexpr int KT = 64;  // keys per tile
// Lazy-reference slack: a lane's tile sum of p above it moves the reference.  2^16, and 2^15
// for f16, whose largest finite value is below 2^16.
template <typename T>
constexpr float kSumMax = std::is_same<T, f16>::value ? 32768.f : 65536.f;

// LDS tiles hold 64 rows (keys) of DH elements, unpadded; 16-byte chunk c of row r sits at
// chunk position kswz / vswz.  K is read 32 rows at one chunk (16 bytes a lane), V 8 rows at
// two neighbouring chunks (8 bytes a lane); each xor spreads its pattern over all banks.
template <int DH>
__device__ __forceinline__ int kswz(int r, int c) {
    return DH == 64 ? c ^ ((r >> 1) & 7) : c ^ (r & 15);
}
template <int DH>
__device__ __forceinline__ int vswz(int r, int c) {
    return DH == 64 ? c ^ (2 * ((r >> 1) & 3)) : c ^ (2 * (r & 7));
}

typedef short i16x4 __attribute__((ext_vector_type(4)));
// Four keys k0 .. k0 + 3 of dim d = 32 db + lane % 32, k0 = base + 4 (lane / 32): within each
// 16-lane group lane i reads 8 bytes of row k0 + i / 4 at dims 16 (group & 1) + 4 (i % 4), and
// the transposing read hands lane j the group's column j.
template <int DH>
__device__ __forceinline__ i16x4 read_v4(const unsigned char* tile, int base, int db, int lane) {
    const int i = lane & 15, grp = lane >> 4;
    const int row = base + 4 * (grp >> 1) + (i >> 2);
    const int col = 32 * db + 16 * (grp & 1) + 4 * (i & 3);  // element; chunk col / 8
    const unsigned char* p = tile + row * (DH * 2) + (vswz<DH>(row, col >> 3) << 4) + (col & 7) * 2;
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)p);
}
// The V^T operand of 16-key group g and dim block db: keys 16 g + 4 h + 0..3, 16 g + 8 + 4 h + 0..3.
template <typename T, int DH>
__device__ __forceinline__ typename Vec8<T>::type read_v(const unsigned char* tile, int g, int db, int lane) {
    struct { i16x4 a, b; } f = {read_v4<DH>(tile, 16 * g, db, lane), read_v4<DH>(tile, 16 * g + 8, db, lane)};
    return __builtin_bit_cast(typename Vec8<T>::type, f);
}

// Raw scores S^T of one tile (two 32-key blocks).
template <typename T, int DH>
__device__ __forceinline__ void score_tile(f32x16 (&s)[2], const unsigned char* kt, int fr, int fh,
                                           const typename Vec8<T>::type (&qf)[DH / 16]) {
    typedef typename Vec8<T>::type V8;
#pragma unroll
    for (int kb = 0; kb < 2; kb++) {
        V8 kf[DH / 16];
        const int r = 32 * kb + fr;
#pragma unroll
        for (int ks = 0; ks < DH / 16; ks++)
            kf[ks] = *reinterpret_cast<const V8*>(kt + r * (DH * 2) + (kswz<DH>(r, 2 * ks + fh) << 4));
        f32x16 z;
#pragma unroll
        for (int e = 0; e < 16; e++) z[e] = 0.f;
        s[kb] = z;
#pragma unroll
        for (int ks = 0; ks < DH / 16; ks++) s[kb] = mma32x16(kf[ks], qf[ks], s[kb]);
    }
}

template <int N>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// The key tiles 64 w .. 64 w + 63 of a row that hold a valid key, compacted in order: lane i
// holds the i-th one's index and its 64-bit key validity.
struct TileWord {
    int t, lo, hi;  // per lane
    int n;          // wave-uniform
};
__device__ __forceinline__ TileWord tile_word(const float* mask, int len, int nt, int w, int lane) {
    const int t0 = 64 * w, g = t0 + lane;
    unsigned long long bits = 0ull;
    if (mask == nullptr) {
        const int rem = len & (KT - 1);
        if (g < nt) bits = (g == nt - 1 && rem) ? (1ull << rem) - 1ull : ~0ull;
    } else {
        const int n = nt - t0 < 64 ? nt - t0 : 64;
        for (int i = 0; i < n; i += 16) {  // 16 tiles' masks in flight
            float mv[16];
#pragma unroll
            for (int u = 0; u < 16; u++) {
                const int key = (t0 + i + u) * KT + lane;
                mv[u] = i + u < n && key < len ? mask[key] : 0.f;
            }
#pragma unroll
            for (int u = 0; u < 16; u++) {
                const unsigned long long m = __ballot(mv[u] >= 0.5f);
                if (lane == i + u) bits = m;
            }
        }
    }
    const bool on = bits != 0ull;
    const unsigned long long act = __ballot(on);
    const int cnt = __popcll(act), below = __popcll(act & ((1ull << lane) - 1ull));
    const int dest = 4 * (on ? below : cnt + (lane - below));
    TileWord tw;
    tw.t = __builtin_amdgcn_ds_permute(dest, g);
    tw.lo = __builtin_amdgcn_ds_permute(dest, (int)(unsigned)bits);
    tw.hi = __builtin_amdgcn_ds_permute(dest, (int)(unsigned)(bits >> 32));
    tw.n = cnt;
    return tw;
}

// 64-dim heads run the scores of tile j + 1 on the matrix cores under the softmax of tile j
// (LOOK), so their K streams one step further ahead than V; 128-dim heads have no registers for
// a second score tile.  Two ring slots: three (96 KB) measured 14.1 against 13.0 us at 1 x 20
// heads x 750 x 950 and 35 against 21 us at 2 x 16 x 750 x 1381, where the second workgroup per
// CU is worth more than the second step of lookahead.
// UNAL: operands off a dword boundary, tiles through registers (the 16-byte loads take any
// address, the buffer-to-LDS ones any dword-aligned address).
template <typename T, int DH, int QB, int KVS, bool UNAL>
__global__ __launch_bounds__(64 * QB * KVS) __attribute__((amdgpu_waves_per_eu(1, 2))) void attn_nv_kernel(
    AttnArgs<T> a, int nqb) {
    typedef typename Vec8<T>::type V8;
    constexpr int NW = QB * KVS, ROWB = DH * 2, TILE = KT * ROWB, RPI = 1024 / ROWB, NI = KT / RPI, RS = 2;
    constexpr int LPW = KVS * NI / NW;  // load instructions per wave per K (or V) stage
    constexpr int KS = DH / 16, DB = DH / 32, CH = DH / 8;
    constexpr bool LOOK = DH == 64;
    static_assert(LPW * NW == KVS * NI, "tiles must split over the waves");
    static_assert((KVS - 1) * QB * (DB * 16 + 2) * 256 <= 2 * RS * KVS * TILE, "merge buffer must fit the rings");
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    unsigned char* kring = smem;                     // [RS][KVS][TILE]
    unsigned char* vring = smem + RS * KVS * TILE;   // [RS][KVS][TILE]

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int qb = wave % QB, par = wave / QB;
    const int pid = xcd_remap(blockIdx.x, gridDim.x);
    const int qblk = pid % nqb, bhid = pid / nqb;
    const int hh = bhid % a.H, b = bhid / a.H;
    const int q = qblk * (32 * QB) + 32 * qb + (lane & 31);
    const int fr = lane & 31, fh = lane >> 5;
    const size_t bh = (size_t)b * a.H + hh;
    const int nt = (a.len0 + KT - 1) / KT;
    const T* Kb = a.K0 + bh * a.stride0 * DH;
    const T* Vb = a.V0 + bh * a.stride0 * DH;
    const float* mb = a.mask0 ? a.mask0 + (size_t)b * a.len0 : nullptr;
    // c = 0 would turn a masked key's -inf into NaN; a tiny c gives the same exp2(0).
    float c = a.scale * 1.4426950408889634f;
    c = c == 0.f ? 1e-38f : c;
    const float s_masked = c > 0.f ? -INFINITY : INFINITY;

    // Load instruction ii of this wave in a stage: gi = wave * LPW + ii -> parity tile gi / NI,
    // rows RPI (gi % NI) ..; lane -> row lane / CH, physical chunk lane % CH.
    unsigned voK[LPW], voV[LPW];
#pragma unroll
    for (int ii = 0; ii < LPW; ii++) {
        const int r = ((wave * LPW + ii) % NI) * RPI + lane / CH;
        voK[ii] = (unsigned)(r * ROWB + (kswz<DH>(r, lane % CH) << 4));
        voV[ii] = (unsigned)(r * ROWB + (vswz<DH>(r, lane % CH) << 4));
    }

    V8 qf[KS];
    {
        const T* qp = a.Q + (bh * a.Sq + (q < a.Sq ? q : a.Sq - 1)) * DH + 8 * fh;
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
            qf[ks] = __builtin_bit_cast(V8, *reinterpret_cast<const u32x4_u*>(qp + 16 * ks));
    }
    f32x16 o[DB];
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
        for (int e = 0; e < 16; e++) o[db][e] = 0.f;
    float m = 0.f, l_run = 0.f;
    bool unset = true;  // m is no reference yet: no tile so far, or only scores of -inf
    bool first = true;  // any lane's unset

    for (int w = 0; 64 * w < nt; w++) {  // 4096 keys at a time
        const TileWord tw = tile_word(mb, a.len0, nt, w, lane);
        const int nact = tw.n, niter = (nact + KVS - 1) / KVS;
        if (niter == 0) continue;  // the same for every wave
        if (w > 0) {               // the rings are still being read
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            raw_barrier();
        }
        // K (or V) tiles of step j into ring slot `slot`.  Entries past the last are clamped to
        // it, so every wave issues LPW loads per stage.
        auto issue = [&](bool is_v, int j, int slot) {
#pragma unroll
            for (int ii = 0; ii < LPW; ii++) {
                const int gi = wave * LPW + ii;
                int li = j * KVS + gi / NI;
                li = li < nact ? li : nact - 1;
                const int t = __builtin_amdgcn_readlane(tw.t, li);
                const T* src = (is_v ? Vb : Kb) + (size_t)t * KT * DH;
                const int rows = a.len0 - t * KT;  // (of every key left, the window's bytes would wrap at 4 GiB)
                const unsigned bytes = (unsigned)(rows < KT ? rows : KT) * (unsigned)ROWB;
                const unsigned vo = is_v ? voV[ii] : voK[ii];
                unsigned char* dst = (is_v ? vring : kring) + (slot * KVS + gi / NI) * TILE + (gi % NI) * 1024;
                if constexpr (UNAL) {
                    u32x4 x = {0, 0, 0, 0};
                    if (vo < bytes) x = *reinterpret_cast<const u32x4_u*>(src + vo / 2);  // whole rows in or out
                    *reinterpret_cast<u32x4*>(dst + 16 * lane) = x;
                } else {
                    buf_load_lds16(make_rsrc(src, bytes), vo, dst);
                }
            }
        };
        issue(false, 0, 0);
        issue(true, 0, 0);
        f32x16 s[2], sn[2];
        if constexpr (LOOK) {
            if (niter > 1) {
                issue(false, 1, 1);
                wait_loads<2 * LPW>();
            } else {
                wait_loads<0>();
            }
            if constexpr (UNAL) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the tiles' LDS writes
            raw_barrier();
            if (par < nact) score_tile<T, DH>(s, kring + par * TILE, fr, fh, qf);
        }

        // Tile step j consumes sc (its raw scores; computed here without LOOK) and leaves tile
        // j + 1's in sx.
        auto tile_step = [&](int j, f32x16 (&sc)[2], f32x16 (&sx)[2]) {
            // This wave's loads of V_j and K_{j+1} (K_j) have landed, and its LDS reads of step
            // j - 1 are done, whose slots are refilled after the barrier.
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            raw_barrier();
            if (j + 1 < niter) issue(true, j + 1, (j + 1) & 1);
            if (j + 1 + LOOK < niter) issue(false, j + 1 + LOOK, (j + 1 + LOOK) & 1);
            const int li = j * KVS + par;
            if (li >= nact) return;  // this parity has no tile in the last step
            const int slot = j & 1;
            const unsigned char* vt = vring + (slot * KVS + par) * TILE;
            if constexpr (!LOOK) score_tile<T, DH>(sc, kring + (slot * KVS + par) * TILE, fr, fh, qf);
            V8 vf[DH == 64 ? 2 : 1][4];
            if constexpr (DH == 64) {  // read now: their latency hides behind the softmax
#pragma unroll
                for (int db = 0; db < 2; db++)
#pragma unroll
                    for (int g = 0; g < 4; g++) vf[db][g] = read_v<T, DH>(vt, g, db, lane);
            }
            const unsigned blo = (unsigned)__builtin_amdgcn_readlane(tw.lo, li);
            const unsigned bhi = (unsigned)__builtin_amdgcn_readlane(tw.hi, li);
            if ((blo & bhi) != 0xffffffffu) {  // keys 32 kb + 8 g4 + 4 fh + i of this lane
#pragma unroll
                for (int kb = 0; kb < 2; kb++) {
                    const unsigned wd = (kb ? bhi : blo) >> (4 * fh);
#pragma unroll
                    for (int g4 = 0; g4 < 4; g4++)
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            if (!((wd >> (8 * g4 + i)) & 1u)) sc[kb][4 * g4 + i] = s_masked;
                }
            }
            // Largest scaled score of the query over the tile, above the reference sub.
            auto tile_max = [&](float sub) {
                float mx[16];
#pragma unroll
                for (int e = 0; e < 16; e++) mx[e] = fmaxf(fmaf(sc[0][e], c, -sub), fmaf(sc[1][e], c, -sub));
#pragma unroll
                for (int h = 8; h > 0; h >>= 1)
#pragma unroll
                    for (int e = 0; e < h; e++) mx[e] = fmaxf(mx[e], mx[e + h]);
                return max_halves(mx[0]);
            };
            if (first) {
                // (A query whose scores are all -inf so far adds nothing at any m, and must not keep
                // one: scores far below it would vanish.)
                const float t = tile_max(0.f);
                if (unset && t != -INFINITY) {
                    m = t;
                    unset = false;
                }
                first = __any(unset);
            }
            if constexpr (LOOK) score_tile<T, DH>(sx, kring + (((j + 1) & 1) * KVS + par) * TILE, fr, fh, qf);
            float psum = 0.f;
            V8 pf[4];
#pragma unroll
            for (int kb = 0; kb < 2; kb++)
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const float p = fast_exp2(fmaf(sc[kb][e], c, -m));
                    psum += p;
                    pf[2 * kb + (e >> 3)][e & 7] = static_cast<T>(p);
                }
            if constexpr (LOOK) {  // the next tile's K reads, then its MFMAs spread over the softmax
                __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 14, 0);
                }
            }
            const unsigned long long over = __ballot(!(psum <= kSumMax<T>));
            if (over) {
                // Lanes l and l ^ 32 hold one query's two key halves: either one asks for both.
                const bool need = ((over >> lane) | (over >> (lane ^ 32))) & 1ull;
                const float mx = tile_max(m);
                const float nm = need ? m + mx : m, corr = fast_exp2(m - nm);
                m = nm;
#pragma unroll
                for (int db = 0; db < DB; db++) o[db] *= corr;
                l_run *= corr;
                psum = 0.f;
#pragma unroll
                for (int kb = 0; kb < 2; kb++)
#pragma unroll
                    for (int e = 0; e < 16; e++) {
                        const float p = fast_exp2(fmaf(sc[kb][e], c, -m));
                        psum += p;
                        pf[2 * kb + (e >> 3)][e & 7] = static_cast<T>(p);
                    }
            }
            l_run += psum;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    if constexpr (DH == 64) o[db] = mma32x16(vf[db][g], pf[g], o[db]);
                    else o[db] = mma32x16(read_v<T, DH>(vt, g, db, lane), pf[g], o[db]);
                }
        };
        for (int j = 0; j < niter; j += 2) {
            tile_step(j, s, sn);
            if (j + 1 < niter) tile_step(j + 1, sn, s);
        }
    }

    // Merge the key parities through LDS [parity - 1][QB][16 DB + 2][64 lanes] in parity order.
    if constexpr (KVS > 1) {
        float m_run = unset ? -INFINITY : m;
        float* comb = reinterpret_cast<float*>(smem) + lane;
        constexpr int PER = (16 * DB + 2) * 64;
        __syncthreads();
        if (par > 0) {
            float* cp = comb + ((par - 1) * QB + qb) * PER;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int e = 0; e < 16; e++) cp[(16 * db + e) * 64] = o[db][e];
            cp[16 * DB * 64] = m_run;
            cp[(16 * DB + 1) * 64] = l_run;
        }
        __syncthreads();
        if (par > 0) return;
#pragma unroll
        for (int pp = 1; pp < KVS; pp++) {
            const float* cp = comb + ((pp - 1) * QB + qb) * PER;
            const float m1 = cp[16 * DB * 64], l1 = cp[(16 * DB + 1) * 64];
            const float mt = fmaxf(m_run, m1), mu = mt == -INFINITY ? 0.f : mt;
            const float c0 = fast_exp2(m_run - mu), c1 = fast_exp2(m1 - mu);
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int e = 0; e < 16; e++) o[db][e] = o[db][e] * c0 + cp[(16 * db + e) * 64] * c1;
            l_run = l_run * c0 + l1 * c1;
            m_run = mt;
        }
    }

    // o[db][e] = O[q][32 db + 8 (e / 4) + 4 fh + e % 4].
    const float l = sum_halves(l_run);
    const float inv = l > 0.f ? 1.f / l : 0.f;
    if (q >= a.Sq) return;
    if (a.out_mode == 0) {
        typedef T T4 __attribute__((ext_vector_type(4)));
        const size_t base = ((size_t)b * a.Sq + q) * ((size_t)a.H * DH) + hh * DH + 4 * fh;
        T4 g[DB][4];
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int g4 = 0; g4 < 4; g4++) g[db][g4] = *reinterpret_cast<const T4*>(a.G + base + 32 * db + 8 * g4);
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int g4 = 0; g4 < 4; g4++) {
                T4 ov;
#pragma unroll
                for (int i = 0; i < 4; i++)
                    ov[i] = static_cast<T>(o[db][4 * g4 + i] * inv * static_cast<float>(g[db][g4][i]));
                *reinterpret_cast<T4*>(a.O + base + 32 * db + 8 * g4) = ov;
            }
    } else {
        float* op = a.Of + (bh * a.Sq + q) * DH + 4 * fh;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int g4 = 0; g4 < 4; g4++)
                store4u(op + 32 * db + 8 * g4, o[db][4 * g4] * inv, o[db][4 * g4 + 1] * inv, o[db][4 * g4 + 2] * inv,
                        o[db][4 * g4 + 3] * inv);
    }
}

template <int DH, int KVS>
constexpr int kLds = 4 * KVS * KT * DH * 2;
template <typename T, int DH, int QB, int KVS, bool UNAL>
hipError_t set_limit() {
    static LdsLimit lim;
    return set_lds_limit_once(lim, (const void*)attn_nv_kernel<T, DH, QB, KVS, UNAL>, kLds<DH, KVS>);
}
template <typename T, int DH, int QB, int KVS, bool UNAL = false>
int launch_cfg(const AttnArgs<T>& a, hipStream_t st) {
    if (set_limit<T, DH, QB, KVS, UNAL>() != hipSuccess) return -2;
    const long wgs = (long)((a.Sq + 32 * QB - 1) / (32 * QB)) * a.H * a.B;
    if (wgs > 0x7fffffffL) return -1;
    attn_nv_kernel<T, DH, QB, KVS, UNAL>
        <<<(unsigned)wgs, 64 * QB * KVS, kLds<DH, KVS>, st>>>(a, (a.Sq + 32 * QB - 1) / (32 * QB));
    return 0;
}
// Every variant that launch_attention_nv<T, DH> chooses from.
template <typename T, int DH>
hipError_t set_limits() {
    hipError_t e = set_limit<T, DH, 2, 2, false>();
    if (e == hipSuccess) e = set_limit<T, DH, 2, 2, true>();
    if (DH == 128 && e == hipSuccess) e = set_limit<T, DH, 4, 2, false>();
    return e;
}

}  // namespace

// Two query blocks and two key parities (64 KB of LDS for 64-dim heads, two workgroups per CU;
// 128 KB for 128-dim heads).  Launches of 128-dim heads that fill most of the chip with twice
// the query blocks per workgroup take four: 31.6 against 46.5 us at 2 x 16 heads x 700 x 1400
// (192 workgroups), but 13.6 against 11.3 at 1 x 10 x 375 x 375 (30).  64-dim heads lose with
// four at every size measured (16.6 against 13.2 us at 1 x 20 x 750 x 950).  A query block's
// arithmetic is the same in either.  The line of UNAL is what the buffer-to-LDS loads take: at 1 x
// 20 x 750 x 950 operands on a dword boundary take 13.1 us (64-dim) and 18.3 (128-dim) as 16-byte
// aligned ones do, through registers 20.5 and 33.4.
template <typename T, int DH>
int launch_attention_nv(const AttnArgs<T>& a, hipStream_t st) {
    if (a.Sq <= 0 || a.len0 <= 0 || a.K1 || a.v_transposed || a.prescaled) return -1;
    if (a.out_mode == 0 ? (!a.G || !a.O) : !a.Of) return -1;
    if ((reinterpret_cast<uintptr_t>(a.Q) | reinterpret_cast<uintptr_t>(a.K0) | reinterpret_cast<uintptr_t>(a.V0)) & 3)
        return launch_cfg<T, DH, 2, 2, true>(a, st);
    if (DH == 128 && (long)((a.Sq + 127) / 128) * a.H * a.B >= 160) return launch_cfg<T, DH, 4, 2>(a, st);
    return launch_cfg<T, DH, 2, 2>(a, st);
}

template int launch_attention_nv<bf16, 64>(const AttnArgs<bf16>&, hipStream_t);
template int launch_attention_nv<bf16, 128>(const AttnArgs<bf16>&, hipStream_t);
template int launch_attention_nv<f16, 64>(const AttnArgs<f16>&, hipStream_t);
template int launch_attention_nv<f16, 128>(const AttnArgs<f16>&, hipStream_t);

hipError_t prepare_attention_nv() {
    hipError_t e = set_limits<bf16, 64>();
    if (e == hipSuccess) e = set_limits<bf16, 128>();
    if (e == hipSuccess) e = set_limits<f16, 64>();
    if (e == hipSuccess) e = set_limits<f16, 128>();
    return e;
}

}  // namespace irodori
