// Kernels of the learned warm start: a 3-D convolutional U-Net that maps a pore geometry
// (solid mask + signed distance) to an initial flow field.  No counterpart in the reference
// (its initial state is u = 0, src/Init_multiphase.cpp:569-572); the network output feeds
// the equilibrium initialisation (mflbm_init_equilibrium).
//
// Tensors are channels-last: [D][H][W][C], C a multiple of 8 for bf16 operands so that one
// lane fetches 8 consecutive channels in one 16-byte load.  Every convolution is 3x3x3,
// stride 1, zero padding 1, computed as an implicit GEMM on the MFMA units with bf16
// operands and fp32 accumulation (v_mfma_f32_16x16x32_bf16):
//   forward   Y[m][n] = sum_k A[m][k] B[k][n],  m = voxel, n = output channel,
//             k = tap * Cin + ci, A[m][k] = X[m + off(tap)][ci], B[k][n] = W[n][k];
//   data grad the same kernel on dY with the weights re-laid out as W'[ci][tap' * Cout + co]
//             = W[co][(26 - tap') * Cin + ci] (off(26 - t) = -off(t));
//   weight grad dW[n][k] = sum_m dZ[m][n] A[m][k], the voxel sum split into chunks whose fp32
//             partial tiles are added in chunk order (deterministic).
// Weights are kept as W[n][k] with n padded to 16 and k to 32 (zero padding), fp32 master
// copy plus a bf16 copy for the MFMA operands.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cstdint>
#include <mutex>
#include <type_traits>

#include "../../include/mfnn.h"
#include "conv_plan.h"
#include "device_lock.h"

namespace {

using namespace mfnn;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(__bf16 v) { return (float)v; }

// Workgroup barrier for data exchanged through LDS only: unlike __syncthreads() it leaves the
// loads from memory in flight.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// 16-byte load through a buffer descriptor: a lane past the descriptor's bytes reads zeros, so
// the zero padding of a convolution costs no select (num = 0 for a whole plane outside the
// grid, NOWHERE as the offset of a single lane).  Descriptors address less than 2^31 bytes.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, uint32_t num) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)num, 0x00027000);
}
__device__ __forceinline__ bf16x8 buffer_load16(__amdgpu_buffer_rsrc_t rsrc, uint32_t offset, uint32_t uniform_offset) {
    return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)offset, (int)uniform_offset, 0));
}

// Taps: 0..26, x fastest (dx = tap % 3 - 1, dy = tap / 3 % 3 - 1, dz = tap / 9 - 1); a tap
// outside the grid reads zero (zero padding).

__device__ __forceinline__ int quot(int n, const FastDiv& f) { return (int)(__umulhi((uint32_t)n, f.mul) + ((uint32_t)n & f.one)); }

// Epilogue of a convolution: bias, then ReLU or the gate, stored as bf16 and/or fp32, for four
// consecutive channels n .. n + 3 of voxel mm per call.  quad: cout is a multiple of 4 and every
// pointer is aligned for four values.
struct Epilogue {
    const float* bias;
    const __bf16* gate;
    __bf16* yb;
    float* yf;
    int cout, relu, quad;

    __device__ __forceinline__ f32x4 bias4(int n) const {
        f32x4 b = f32x4{0.f, 0.f, 0.f, 0.f};
        if (bias) {
            if (quad) {
                if (n < cout) b = *reinterpret_cast<const f32x4*>(bias + n);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (n + j < cout) b[j] = bias[n + j];
            }
        }
        return b;
    }
    // the bf16 output of quads: the network's layers
    template <bool RELU, bool GATE>
    __device__ __forceinline__ void store_quad(const f32x4& acc, const f32x4& b, int n, int mm) const {
        if (n >= cout) return;
        const int64_t at = (int64_t)mm * cout + n;
        bf16x4 gt, o;
        if (GATE) gt = *reinterpret_cast<const bf16x4*>(gate + at);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float v = acc[j] + b[j];
            if (RELU) v = v > 0.f ? v : 0.f;
            if (GATE && !(bf2f(gt[j]) > 0.f)) v = 0.f;
            o[j] = (__bf16)v;
        }
        *reinterpret_cast<bf16x4*>(yb + at) = o;
    }
    __device__ __forceinline__ void store(const f32x4& acc, const f32x4& b, int n, int mm) const {
        const int64_t at = (int64_t)mm * cout + n;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (n + j >= cout) return;
            float v = acc[j] + b[j];
            if (relu) v = v > 0.f ? v : 0.f;
            if (gate && !(bf2f(gate[at + j]) > 0.f)) v = 0.f;
            if (yb) yb[at + j] = (__bf16)v;
            if (yf) yf[at + j] = v;
        }
    }
    // calls put(store) with the store that fits this launch
    template <class F>
    __device__ __forceinline__ void each(F&& put) const {
        if (quad && yb && !yf) {
            if (gate && relu) put([this](const f32x4& a, const f32x4& b, int n, int mm) { store_quad<true, true>(a, b, n, mm); });
            else if (gate) put([this](const f32x4& a, const f32x4& b, int n, int mm) { store_quad<false, true>(a, b, n, mm); });
            else if (relu) put([this](const f32x4& a, const f32x4& b, int n, int mm) { store_quad<true, false>(a, b, n, mm); });
            else put([this](const f32x4& a, const f32x4& b, int n, int mm) { store_quad<false, false>(a, b, n, mm); });
        } else if (quad && yf && !yb && !gate && !relu) {
            put([this](const f32x4& a, const f32x4& b, int n, int mm) {
                if (n >= cout) return;
                f32x4 v;
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = a[j] + b[j];
                *reinterpret_cast<f32x4*>(yf + (int64_t)mm * cout + n) = v;
            });
        } else {
            put([this](const f32x4& a, const f32x4& b, int n, int mm) { store(a, b, n, mm); });
        }
    }
};

// Forward / data-gradient convolution on boxes of voxels staged through LDS.  A workgroup of
// four waves owns tx x ty x tz voxels, numbered x fastest and cut into 16-voxel MFMA tiles,
// MT of them per wave, and the 16-channel tiles blockIdx.y * NT .. + NT - 1.  It loads its box
// with a one-voxel halo once, zeros outside the grid, and every tap of every voxel is then an
// LDS read at the voxel's place plus an offset common to all voxels (s_tab: per 8-channel
// piece of k).  In LDS a piece is an array over the box's voxels, padded to whole rounds of
// the banks: a 16-byte read serves 16 lanes at a time, half of them of one k group of the
// MFMA operand and half of the next, and with even and odd pieces a multiple of 256 bytes
// apart the 16 neighbours in x meet 16 different bank groups; pairs of pieces are skewed by
// one unit for the stores.  The weights go through LDS too, four k blocks at a time: each wave
// loads the operands of one of the four, PF chunks ahead in registers, and all waves read
// them (loaded by every wave for itself they were the bound: 7-8 TB/s out of L2 at every size).
// The operands go in as (weights, voxels), so that a lane ends with four consecutive channels
// of one voxel and stores them as one vector.  Every accumulator sums the k blocks in
// ascending order, as k_conv3 does.  Measured launch to launch against a wave per one or two
// tiles that gathered every operand from global memory, in us: 64^3 16 -> 16 channels 28.4 to
// 11.0, 48 -> 16 73.5 to 25.2; 16^3 192 -> 64 55.5 to 12.7; 8^3 128 -> 128 35.2 to 9.1; 128^3
// 48 -> 16 555 to 175 (LDS operand reads, 82 us of it, and the load of 2.5 times the input).
template <int MT, int NT, int PF>
__global__ __launch_bounds__(256) void k_conv3_box(const __bf16* __restrict__ X, const __bf16* __restrict__ Wb, Grid3 g,
                                                   int cin, int kp, int ntw, Epilogue ep, ConvTile t) {
    // 16 zero bytes, the box, the weights of two chunks, s_tab
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, q = lane >> 4;
    const int c8 = cin >> 3, K8 = 27 * c8, LX = t.tx + 2, LY = t.ty + 2, LZ = t.tz + 2;
    auto unit = [&](int ci) { return (ci >> 1) * (2 * t.pv + 1) + (ci & 1) * t.pv; };  // of piece ci, voxel 0
    unsigned char* s_w = smem + 16 * (1 + (c8 + 1) / 2 * (2 * t.pv + 1));
    int* s_tab = reinterpret_cast<int*>(s_w + 2 * 4 * NT * 1024);
    const int nkb = (K8 + 3) >> 2;    // k blocks of 32 = four pieces of 8
    const int nch = (nkb + 3) >> 2;   // chunks of four k blocks
    // boxes in launch order, all of them once per channel group (one contiguous run of boxes
    // per XCD measured up to 6 % slower)
    int bx, by, bz, tb;
    {
        const int b = blockIdx.x, yz = quot(b, t.dnx);
        tb = blockIdx.y * NT;
        bz = quot(yz, t.dny);
        bx = b - yz * t.nx;
        by = yz - bz * t.ny;
    }
    const int x0 = bx * t.tx, y0 = by * t.ty, z0 = bz * t.tz;

    // first weight operands: in flight while the box loads
    const __amdgpu_buffer_rsrc_t wbuf = buffer_of(Wb, 32u * ntw * kp);
    uint32_t wrow[NT];  // byte offset of this lane's operand in this wave's block of chunk 0
#pragma unroll
    for (int n = 0; n < NT; ++n) wrow[n] = 2u * ((min(tb + n, ntw - 1) * 16 + r) * kp + 8 * q + 32 * wave);
    bf16x8 w[PF][NT];
    auto load_w = [&](int slot, int c) {  // zeros past the last k block
        const bool in = 4 * c + wave < nkb;
#pragma unroll
        for (int n = 0; n < NT; ++n) w[slot][n] = buffer_load16(wbuf, in ? wrow[n] : NOWHERE, 256u * c);
    };
    unsigned char* const w_mine = s_w + wave * NT * 1024 + 16 * lane;
    const unsigned char* const w_all = s_w + 16 * lane;
    auto keep_w = [&](int slot) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
            *reinterpret_cast<bf16x8*>(w_mine + ((slot & 1) * 4 * NT + n) * 1024) = w[slot][n];
    };
#pragma unroll
    for (int s = 0; s < PF; ++s) load_w(s, s);

    bf16x8 zero;
#pragma unroll
    for (int j = 0; j < 8; ++j) zero[j] = (__bf16)0.f;
    if (tid == 0) *reinterpret_cast<bf16x8*>(smem) = zero;
    // The box, up to six planes at a time: a thread keeps its place (row, voxel, piece) over the
    // planes and loads its next place's planes before it stores the present one's.
    const uint32_t plane = 2u * g.H * g.W * cin;  // bytes
    constexpr int ZB = 6;
    for (int lz0 = 0; lz0 < LZ; lz0 += ZB) {
        bf16x8 v[2][ZB];
        unsigned char* dst[2];
        auto fetch = [&](int slot, int i) {
            const int ly = quot(i, t.row), c = i - ly * (int)t.row.d;
            const int lx = quot(c, t.c8), ci = c - lx * c8;
            const int xx = x0 + lx - 1, yy = y0 + ly - 1;
            const bool in = i < t.pu && xx >= 0 && yy >= 0 && xx < g.W && yy < g.H;
            const uint32_t src = in ? 2u * ((yy * g.W + xx) * cin + 8 * ci) : NOWHERE;
            dst[slot] = smem + 16 * (1 + ly * LX + lx + unit(ci));
#pragma unroll
            for (int m = 0; m < ZB; ++m) {
                const int zz = z0 + lz0 + m - 1;
                const bool zin = lz0 + m < LZ && zz >= 0 && zz < g.D;
                v[slot][m] = buffer_load16(buffer_of(X + (int64_t)(zin ? zz : 0) * (plane >> 1), zin ? plane : 0u), src, 0);
            }
        };
        auto keep = [&](int slot, int i) {
            if (i < t.pu) {
#pragma unroll
                for (int m = 0; m < ZB; ++m)
                    if (lz0 + m < LZ) *reinterpret_cast<bf16x8*>(dst[slot] + 16 * (lz0 + m) * LX * LY) = v[slot][m];
            }
        };
        fetch(0, tid);
        for (int i0 = 0; i0 < t.pu; i0 += 512) {
            if (i0 + 256 < t.pu) fetch(1, i0 + 256 + tid);
            keep(0, i0 + tid);
            if (i0 + 512 < t.pu) fetch(0, i0 + 512 + tid);
            if (i0 + 256 < t.pu) keep(1, i0 + 256 + tid);
        }
    }
    // byte offsets of the k pieces, -1 past the last tap
    for (int c = tid; c < 16 * nch + 16; c += 256) {
        int off = -1;
        if (c < K8) {
            const int tap = quot(c, t.c8), ci = c - tap * c8;
            const int oz = tap / 9, oy = tap / 3 - 3 * oz, ox = tap % 3;
            off = 16 * ((oz * LY + oy) * LX + ox + unit(ci));
        }
        s_tab[c] = off;
    }
    // this lane's voxel of each tile: its place in LDS
    int base[MT];
#pragma unroll
    for (int u = 0; u < MT; ++u) {
        const int v = min((wave * MT + u) * 16 + r, t.tv - 1);  // past the box: its last voxel, not stored
        const int yz = quot(v, t.dtx), lx = v - yz * t.tx, lz = quot(yz, t.dty), ly = yz - lz * t.ty;
        base[u] = 16 * (1 + (lz * LY + ly) * LX + lx);
    }
    f32x4 acc[MT][NT];
#pragma unroll
    for (int u = 0; u < MT; ++u)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[u][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    keep_w(0);
    lds_barrier();

    // Operands run one k block ahead of the MFMAs and the voxels' offsets two; the scheduling
    // barriers keep the reads of the next block in front of the MFMAs of this one (left to
    // itself the compiler makes every MFMA wait for its own read).  An offset is read before
    // the operands of its block, so that waiting for it waits for none of them.
    bf16x8 a[2][MT], b[2][NT];
    auto read_ab = [&](int slot, int half, int s, int off, bool padded) {
        const int keep = padded ? ~(off >> 31) : ~0;  // past the last tap: the zeros at 0
#pragma unroll
        for (int u = 0; u < MT; ++u) a[slot][u] = *reinterpret_cast<const bf16x8*>(smem + ((base[u] + off) & keep));
#pragma unroll
        for (int n = 0; n < NT; ++n)
            b[slot][n] = *reinterpret_cast<const bf16x8*>(w_all + ((half * 4 + s) * NT + n) * 1024);
    };
    const int* tab = s_tab + q;
    int off[2] = {tab[4], tab[8]};  // of the next two blocks
    read_ab(0, 0, 0, tab[0], true);
    // block s of the chunk whose weights are in `half` of s_w; tab: the chunk's offsets
    auto block = [&](int half, int s, const int* tab, bool padded) {
        if (s == 3) lds_barrier();  // the next chunk's weights are written, this one's are read
        const int next = tab[4 * (s + 3)];
        read_ab((s + 1) & 1, s == 3 ? half ^ 1 : half, (s + 1) & 3, off[0], padded);
        off[0] = off[1];
        off[1] = next;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < MT; ++u)
#pragma unroll
            for (int n = 0; n < NT; ++n)
                acc[u][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[s & 1][n], a[s & 1][u], acc[u][n], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    static_assert(PF % 2 == 0, "slot d's chunk goes to half d & 1");
    int c0 = 0;
    for (; c0 + PF < nch; c0 += PF, tab += 16 * PF)
#pragma unroll
        for (int d = 0; d < PF; ++d) {
            // slot d held chunk c0 + d, already in LDS; the next chunk goes to the other half
            load_w(d, c0 + d + PF);
            keep_w((d + 1) % PF);
#pragma unroll
            for (int s = 0; s < 4; ++s) block(d & 1, s, tab + 16 * d, s == 3);  // only the next chunk may be padded
        }
#pragma unroll
    for (int d = 0; d < PF; ++d)  // the ring holds the chunks left
        if (c0 + d < nch) {
            keep_w((d + 1) % PF);
#pragma unroll
            for (int s = 0; s < 4; ++s) block(d & 1, s, tab + 16 * d, true);
        }
    f32x4 bias4[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) bias4[n] = ep.bias4((tb + n) * 16 + 4 * q);
    ep.each([&](auto&& store) {
#pragma unroll
        for (int u = 0; u < MT; ++u) {
            const int v = (wave * MT + u) * 16 + r;
            const int yz = quot(v, t.dtx), lz = quot(yz, t.dty);
            const int xx = x0 + v - yz * t.tx, yy = y0 + yz - lz * t.ty, zz = z0 + lz;
            if (v >= t.tv || xx >= g.W || yy >= g.H || zz >= g.D) continue;
            const int mm = (zz * g.H + yy) * g.W + xx;
#pragma unroll
            for (int n = 0; n < NT; ++n) store(acc[u][n], bias4[n], (tb + n) * 16 + 4 * q, mm);
        }
    });
}

// The convolution of planes of 2 GiB and more and of channel counts whose boxes do not fit LDS or
// hold too few voxels to pay (from 512 on; conv_plan): every tap gathered from global memory.  One wave per MT tiles of 16 voxels and the
// NT 16-channel tiles blockIdx.y * NT ..: the voxel tiles share each weight load, the channel
// tiles each voxel load.
template <int NT, int MT>
__global__ __launch_bounds__(256) void k_conv3(const __bf16* __restrict__ X, const __bf16* __restrict__ Wb, Grid3 g,
                                               int cin, int kp, int ntw, Epilogue ep) {
    const int M = g.D * g.H * g.W;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m0 = (blockIdx.x * 4 + wave) * 16 * MT;
    if (m0 >= M) return;
    const int r = lane & 15, q = lane >> 4;
    const int K = 27 * cin, tb = blockIdx.y * NT;
    int mv[MT], xv[MT], yv[MT], zv[MT];
#pragma unroll
    for (int u = 0; u < MT; ++u) {
        mv[u] = m0 + 16 * u + r;
        xv[u] = mv[u] % g.W;
        yv[u] = (mv[u] / g.W) % g.H;
        zv[u] = mv[u] / (g.W * g.H);
    }
    f32x4 acc[MT][NT];
#pragma unroll
    for (int u = 0; u < MT; ++u)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int kb = 0; kb < kp; kb += 32) {
        const int k = kb + 8 * q;
        const int tap = k < K ? k / cin : 0, ci = k - tap * cin;
        const int ox = tap % 3 - 1, oy = (tap / 3) % 3 - 1, oz = tap / 9 - 1;
        bf16x8 b[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t)
            b[t] = *reinterpret_cast<const bf16x8*>(Wb + (int64_t)((NT == 1 ? tb : min(tb + t, ntw - 1)) * 16 + r) * kp + k);
#pragma unroll
        for (int u = 0; u < MT; ++u) {
            bf16x8 a;
#pragma unroll
            for (int j = 0; j < 8; ++j) a[j] = (__bf16)0.f;
            const int xx = xv[u] + ox, yy = yv[u] + oy, zz = zv[u] + oz;
            if (k < K && mv[u] < M && xx >= 0 && yy >= 0 && zz >= 0 && xx < g.W && yy < g.H && zz < g.D)
                a = *reinterpret_cast<const bf16x8*>(X + (int64_t)((zz * g.H + yy) * g.W + xx) * cin + ci);
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[t], a, acc[u][t], 0, 0, 0);
        }
    }
    auto store_all = [&](auto&& store) {
#pragma unroll
        for (int u = 0; u < MT; ++u)
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int n = (tb + t) * 16 + 4 * q;
                if (mv[u] < M) store(acc[u][t], ep.bias4(n), n, mv[u]);
            }
    };
    // one tile: its four stores are too few to choose between forms for
    if (MT * NT == 1) store_all([&ep](const f32x4& a, const f32x4& b, int n, int mm) { ep.store(a, b, n, mm); });
    else ep.each(store_all);
}

// Weight gradient partials where k_conv3_wgrad_rows cannot address its operands (2 GiB and more) or
// does not pay (rows_pay).  Block (kt, nt, chunk): one wave per 16 x 16·KT block of (output channel
// n, k) over `chunk` voxels, as KT 16 x 16 MFMA tiles that share the dZ operand; writes
// part[chunk][n][k] (fp32).  The waves of the first k block also sum the dZ values they load: the
// bias gradient partials bpart[chunk][n] (n < cout; null: not wanted).
// Per step of 32 voxels the operands are staged through LDS: lane (v, h) loads 8 channels
// (16 bytes) of voxel v -- dZ channels n0 + 8h .., and of each tile the 8 columns
// k0 + 16t + 8h .. (8 consecutive channels of one tap, since cin is a multiple of 8) at the
// tap's shifted voxel -- and lane (r, q) then reads column r of voxels 8q .. 8q + 7, the
// MFMA operand layout.
template <int KT>
__global__ __launch_bounds__(64) void k_conv3_wgrad(const __bf16* __restrict__ X, const __bf16* __restrict__ dZ,
                                                    Grid3 g, int cin, int kp, int coutp, int cout, int chunk,
                                                    float* __restrict__ part, float* __restrict__ bpart) {
    __shared__ __attribute__((aligned(16))) __bf16 sA[32][16];
    __shared__ __attribute__((aligned(16))) __bf16 sB[KT][32][16];
    const int M = g.D * g.H * g.W;
    const int lane = threadIdx.x;
    const int k0 = blockIdx.x * 16 * KT, n0 = blockIdx.y * 16, c = blockIdx.z;
    const int r = lane & 15, q = lane >> 4;  // MFMA role: column r, voxels 8q .. 8q + 7
    const int v = lane >> 1, h = lane & 1;   // loader role: voxel v, 8-channel half h
    const int K = 27 * cin;
    const int n = n0 + r;
    const bool ain = n0 + 8 * h < cout;  // cout is a multiple of 8: the whole half or none
    int lci[KT], lox[KT], loy[KT], loz[KT], loff[KT];
    bool lkin[KT];
#pragma unroll
    for (int t = 0; t < KT; ++t) {
        const int kk = k0 + 16 * t + 8 * h;
        lkin[t] = kk < K;  // K is a multiple of 8: the whole half or none
        const int tap = lkin[t] ? kk / cin : 0;
        lci[t] = lkin[t] ? kk - tap * cin : 0;
        lox[t] = tap % 3 - 1;
        loy[t] = (tap / 3) % 3 - 1;
        loz[t] = tap / 9 - 1;
        loff[t] = (loz[t] * g.H + loy[t]) * g.W + lox[t];
    }
    f32x4 acc[KT];
#pragma unroll
    for (int t = 0; t < KT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    float bsum = 0.f;  // this lane's dZ values (row n), in voxel order
    const int mb = c * chunk, me = min(M, mb + chunk);
    bf16x8 zero;
#pragma unroll
    for (int j = 0; j < 8; ++j) zero[j] = (__bf16)0.f;
    for (int ms = mb; ms < me; ms += 32) {
        const int m = ms + v;
        bf16x8 la = zero;
        if (m < me && ain) la = *reinterpret_cast<const bf16x8*>(dZ + (int64_t)m * cout + n0 + 8 * h);
        *reinterpret_cast<bf16x8*>(&sA[v][8 * h]) = la;
        const int x = m % g.W, y = (m / g.W) % g.H, z = m / (g.W * g.H);
#pragma unroll
        for (int t = 0; t < KT; ++t) {
            const int xx = x + lox[t], yy = y + loy[t], zz = z + loz[t];
            const bool in = m < me && lkin[t] && xx >= 0 && yy >= 0 && zz >= 0 && xx < g.W && yy < g.H && zz < g.D;
            bf16x8 lb = zero;
            if (in) lb = *reinterpret_cast<const bf16x8*>(X + (int64_t)(m + loff[t]) * cin + lci[t]);
            *reinterpret_cast<bf16x8*>(&sB[t][v][8 * h]) = lb;
        }
        __syncthreads();
        bf16x8 a, b[KT];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            a[j] = sA[8 * q + j][r];
#pragma unroll
            for (int t = 0; t < KT; ++t) b[t][j] = sB[t][8 * q + j][r];
        }
        if (bpart && k0 == 0) {
#pragma unroll
            for (int j = 0; j < 8; ++j) bsum += bf2f(a[j]);
        }
#pragma unroll
        for (int t = 0; t < KT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[t], acc[t], 0, 0, 0);
        __syncthreads();
    }
    if (bpart && k0 == 0) {
        // lanes r, r + 16, r + 32, r + 48 hold row n: fixed pairing order
        const float s1 = bsum + __shfl_xor(bsum, 16);
        const float s2 = s1 + __shfl_xor(s1, 32);
        if (q == 0 && n < cout) bpart[(int64_t)c * cout + n] = s2;
    }
    // tile t: D[row = n0 + 4q + j][col = k0 + 16t + r]
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) part[((int64_t)c * coutp + n0 + 4 * q + j) * kp + k0 + 16 * t + r] = acc[t][j];
}

// Weight gradient partials with the operands shared through LDS.  A workgroup owns one chunk of
// voxels, one plane offset dz of the taps, a slice of 16 input channels (HALF: the last 8 of an
// odd multiple of 8) and a 16-channel tile of the output; its three waves take the three row
// offsets dy, so that a wave accumulates the three taps of a row (three MFMA tiles, two with two
// 8-channel taps to a tile).  With G = 2 a second group of three waves takes every other block of
// 32 voxels.  Up to `sub` voxels at a time, it loads the rows that
// these voxels' taps reach once, padded by a zero voxel at each end and a zero row above and
// below each plane, and the voxels' dZ; s_pos holds each voxel's place among the rows, from
// which every tap is a fixed distance.  The MFMA operands hold eight voxels of one channel per
// lane: the transposing LDS read (four 16-bit rows per 16 lanes) delivers them from the
// channels-last rows.  Gathered per tap from global memory and transposed by eight 2-byte LDS
// reads per operand (k_conv3_wgrad, one wave per tile) the same sums were bound by those reads
// and by 27-fold loads of the input.  Every accumulator adds the voxel blocks of a chunk in
// ascending order (of each group, whose sums are then added).  Measured with the chunk sums
// against one wave per 16 or 32 columns, in us: 64^3 16 -> 16 channels 82.7 to 25.2, 48 -> 16 127
// to 47; 32^3 96 -> 32 72 to 31.7; 128^3 16 -> 16 317 to 132.  At 64^3 the 64 dependent blocks of a
// chunk and its four stages of loads bound it, at 128^3 the vector instructions of the staging.
// Two output tiles to a workgroup, sharing the rows, measured no faster on any of 17 shapes but
// one once a chunk's workgroups share an XCD (128^3 32 -> 32 390 against 402), and slower on others
// (128^3 16 -> 48 384 against 311, 96^3 24 -> 40 315 against 220).
struct WgradRows {
    int gx, gy, per_xcd; // workgroups of a chunk along the input and the output channels; their order
    int ci0, sub;        // first channel, voxels staged at a time
    int planes;          // a plane holds a stage, and there are several
    int lds_dz, lds_pos; // byte offsets of the staged dZ and of s_pos
    FastDiv row, h2, w, h;  // 16-byte units of a padded row; H + 2, W, H
};

// Place of workgroup b in an order where each of the 8 XCDs takes one contiguous run (workgroups
// go to the XCDs in turn).
__device__ __forceinline__ int contiguous_per_xcd(int total, int b) {
    const int per = total >> 3, rem = total & 7, xcd = b & 7;
    return xcd * per + min(xcd, rem) + (b >> 3);
}

__device__ __forceinline__ bf16x4 read_transposed(const unsigned char* lds) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                          (__attribute__((address_space(3))) s16x4*)const_cast<unsigned char*>(lds)));
}

template <bool HALF, int G>
__global__ __launch_bounds__(192 * G) void k_conv3_wgrad_rows(const __bf16* __restrict__ X, const __bf16* __restrict__ dZ,
                                                          Grid3 g, int cin, int kp, int coutp, int cout, int chunk,
                                                          WgradRows t, float* __restrict__ part,
                                                          float* __restrict__ bpart) {
    // 128 zero bytes, the padded rows, the voxels' dZ, the voxels' places
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    constexpr int VB = HALF ? 16 : 32, PU = VB / 16;  // bytes and units of a voxel
    constexpr int NT = HALF ? 2 : 3;                  // MFMA column tiles of a wave
    int* s_pos = reinterpret_cast<int*>(smem + t.lds_pos);
    constexpr int TH = 192 * G;
    const int tid = threadIdx.x, lane = tid & 63, wave6 = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave6 / 3, wave = wave6 - 3 * grp;
    const int r = lane & 15, q = lane >> 4;
    int slice, dzi, n0, c;
    {
        const int per = t.gx * t.gy, l = t.per_xcd ? contiguous_per_xcd(gridDim.x, blockIdx.x) : blockIdx.x;
        c = l / per;
        const int xy = l - c * per, by = xy / t.gx, bx = xy - by * t.gx;
        n0 = by * 16;
        slice = bx / 3;
        dzi = bx - 3 * slice;
    }
    const int ci0 = t.ci0 + 16 * slice;
    const int M = g.D * g.H * g.W, mb = c * chunk, me = min(M, mb + chunk);
    const int WP = g.W + 2;
    const bool first = slice == 0 && dzi == 0 && t.ci0 == 0;
    const bool bias = bpart && first && wave == 0;
    // this lane's part of the operand reads: voxel r / 4 of four, channels 4 (r % 4) ..; with two
    // taps to a tile the upper quarters read the next voxel of the row (the tile past the third
    // tap is not stored)
    const int lane_off = HALF ? ((r >> 1) & 1) * VB + (r & 1) * 8 : (r & 3) * 8;
    const int tap_off = ((wave - 1) * WP - 1) * VB + lane_off;  // of the row's first tap from the voxel
    constexpr int TSTEP = HALF ? 2 * VB : VB;                   // from one column tile to the next
    f32x4 acc[NT];
#pragma unroll
    for (int u = 0; u < NT; ++u) acc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    float bsum = 0.f;
    bf16x8 zero;
#pragma unroll
    for (int j = 0; j < 8; ++j) zero[j] = (__bf16)0.f;
    if (tid < 8) *reinterpret_cast<bf16x8*>(smem + 16 * tid) = zero;

    // One stage: the padded rows and the dZ of voxels s0 .. e - 1.  The first PX and PD units of
    // a thread are loaded into registers while the stage before is computed; wider rows load
    // the rest when it is stored.
    constexpr int PX = 10 / G, PD = 6 / G;
    bf16x8 vx[PX], vd[PD];
    int s0, e, xa, ya, za, units, vox, dunits, ylast;
    bool flat;  // every voxel of the stage is in plane za, and the rows' last is ylast - 1
    auto stage = [&](int from) {
        s0 = from;
        e = min(me, s0 + t.sub);
        const int ra = s0 / g.W, rb = (e - 1) / g.W, zb = rb / g.H;
        za = ra / g.H;
        xa = s0 - ra * g.W;
        ya = ra - za * g.H;
        flat = t.planes && zb == za;
        ylast = min(g.H, ya + rb - ra + 2);
        units = (rb - ra + 2 * (zb - za) + 3) * WP * PU;
        vox = (e - s0 + 31) & ~31;
        dunits = vox * 2;
    };
    // unit i of the padded rows: its row, and its byte offset in a row of the input (NOWHERE for
    // the padding)
    auto place = [&](int i, int& row, uint32_t& col) {
        row = quot(i, t.row);
        const int u = i - row * WP * PU, x = u / PU - 1;
        col = x >= 0 && x < g.W ? 2u * (x * cin + ci0 + 8 * (u % PU)) : NOWHERE;
    };
    const __amdgpu_buffer_rsrc_t xbuf = buffer_of(X, 2u * M * cin), dbuf = buffer_of(dZ, 2u * M * cout);
    auto row_unit = [&](int i, int row, uint32_t col) {
        const int yp = ya + row, zo = quot(yp, t.h2), y = yp - zo * (g.H + 2) - 1, z = za + zo + dzi - 1;
        const uint32_t from = __umul24(__umul24(z, g.H) + y, 2u * g.W * cin) + col;
        return buffer_load16(xbuf, i < units && (unsigned)y < (unsigned)g.H && (unsigned)z < (unsigned)g.D ? from : NOWHERE, 0);
    };
    auto dz_unit = [&](int i) {
        const int mv = s0 + i / 2, n = n0 + 8 * (i % 2);
        return buffer_load16(dbuf, mv < e && n < cout ? 2u * (mv * cout + n) : NOWHERE, 0);
    };
    // Within a plane the rows of a stage are one run of the input: a unit's offset from the row of
    // the first voxel is fixed over the stages, and one compare says whether the run holds it (the
    // general address takes 20 instructions; 128^3 16 -> 16 142 to 133 us, 48 -> 16 323 to 308).
    // Two groups of waves have half the units each and keep the general places in registers.
    const uint32_t rowbytes = 2u * g.W * cin;
    uint32_t at[PX];
    int prow[G == 1 ? 1 : PX];
    uint32_t pcol[G == 1 ? 1 : PX];
    if (G > 1) {
#pragma unroll
        for (int m = 0; m < PX; ++m) place(tid + TH * m, prow[G == 1 ? 0 : m], pcol[G == 1 ? 0 : m]);
    } else if (t.planes) {
#pragma unroll
        for (int m = 0; m < PX; ++m) {
            int row;
            uint32_t col;
            place(tid + TH * m, row, col);
            at[m] = col == NOWHERE ? NOWHERE : (row - 1) * rowbytes + col;
        }
    }
    auto fetch = [&]() {
        if (G > 1) {
#pragma unroll
            for (int m = 0; m < PX; ++m) vx[m] = row_unit(tid + TH * m, prow[G == 1 ? 0 : m], pcol[G == 1 ? 0 : m]);
        } else if (flat) {
            const int z = za + dzi - 1;
            const bool in = (unsigned)z < (unsigned)g.D;
            const uint32_t first = ya * rowbytes, end = in ? ylast * rowbytes : 0, plane = in ? z * g.H * rowbytes : 0;
#pragma unroll
            for (int m = 0; m < PX; ++m) {
                const uint32_t o = first + at[m];
                vx[m] = buffer_load16(xbuf, o < end ? o : NOWHERE, plane);
            }
        } else {
            int i = tid;
            asm volatile("" : "+v"(i));  // computed here, not kept over the stages in 20 registers
#pragma unroll
            for (int m = 0; m < PX; ++m) {
                int row;
                uint32_t col;
                place(i + TH * m, row, col);
                vx[m] = row_unit(i + TH * m, row, col);
            }
        }
#pragma unroll
        for (int m = 0; m < PD; ++m) vd[m] = dz_unit(tid + TH * m);
    };
    auto keep = [&]() {
        bf16x8 *rows = reinterpret_cast<bf16x8*>(smem + 128), *ds = reinterpret_cast<bf16x8*>(smem + t.lds_dz);
#pragma unroll
        for (int m = 0; m < PX; ++m)
            if (tid + TH * m < units) rows[tid + TH * m] = vx[m];
#pragma unroll
        for (int m = 0; m < PD; ++m)
            if (tid + TH * m < dunits) ds[tid + TH * m] = vd[m];
        for (int i = tid + TH * PX; i < units; i += TH) {
            int row;
            uint32_t col;
            place(i, row, col);
            rows[i] = row_unit(i, row, col);
        }
        for (int i = tid + TH * PD; i < dunits; i += TH) ds[i] = dz_unit(i);
        for (int v = tid; v < vox; v += TH) {
            const int row = quot(xa + v, t.w), zo = quot(ya + row, t.h);  // rows and planes below voxel s0's
            s_pos[v] = s0 + v < e ? 128 + ((row + 2 * zo + 1) * WP + xa + v - row * g.W + 1) * VB : -1;
        }
    };
    const int v0 = 8 * q + (r >> 2);  // and v0 + 4: the voxels this lane reads for its group
    bf16x8 a[2], b[2][NT];
    const unsigned char* const dz_lane = smem + t.lds_dz + v0 * 32 + (r & 3) * 8;
    auto read_ab = [&](int slot, int ms, int p0, int p1) {
        const unsigned char* d = dz_lane + ms * 32;
        const bf16x4 dlo = read_transposed(d), dhi = read_transposed(d + 4 * 32);
        a[slot] = __builtin_shufflevector(dlo, dhi, 0, 1, 2, 3, 4, 5, 6, 7);
        // a voxel past the grid reads the zeros at 0
        const unsigned char *x0 = smem + (p0 >= 0 ? p0 + tap_off : lane_off), *x1 = smem + (p1 >= 0 ? p1 + tap_off : lane_off);
#pragma unroll
        for (int u = 0; u < NT; ++u) {
            const bf16x4 lo = read_transposed(x0 + u * TSTEP), hi = read_transposed(x1 + u * TSTEP);
            b[slot][u] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
    };
    stage(mb);
    fetch();
    for (;;) {
        keep();
        __syncthreads();
        const int blocks = vox >> 5;
        const bool more = e < me;
        if (more) {
            stage(e);
            fetch();
        }
        // group grp takes blocks grp, grp + G, ..; operands run one of its blocks of 32 voxels
        // ahead of the MFMAs, places two
        const int mine = (blocks - grp + G - 1) / G, last = blocks - 1;
        const int* pos = s_pos + v0;
        auto nth = [&](int i) { return min(grp + G * i, last) * 32; };
        int p0 = pos[nth(0)], p1 = pos[nth(0) + 4];
        read_ab(0, nth(0), p0, p1);
        p0 = pos[nth(1)];
        p1 = pos[nth(1) + 4];
        auto block = [&](int slot, int i) {
            const int n0_ = p0, n1_ = p1;
            p0 = pos[nth(i + 2)];
            p1 = pos[nth(i + 2) + 4];
            read_ab(slot ^ 1, nth(i + 1), n0_, n1_);
            __builtin_amdgcn_sched_barrier(0);
            if (bias) {
#pragma unroll
                for (int j = 0; j < 8; ++j) bsum += bf2f(a[slot][j]);
            }
#pragma unroll
            for (int u = 0; u < NT; ++u)
                acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[slot], b[slot][u], acc[u], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        for (int i = 0; i < mine; i += 2) {
            block(0, i);
            if (i + 1 < mine) block(1, i + 1);
        }
        if (!more) break;
        lds_barrier();  // every wave is done with the stage; the loads of the next stay in flight
    }
    if (G > 1) {
        // the second group's sums are added to the first's
        __syncthreads();
        f32x4* const sum = reinterpret_cast<f32x4*>(smem) + wave * 64 * NT + lane;
        float* const bs = reinterpret_cast<float*>(smem + 3 * 64 * NT * 16) + lane;
        if (grp == 1) {
#pragma unroll
            for (int u = 0; u < NT; ++u) sum[u * 64] = acc[u];
            if (bias) bs[0] = bsum;
        }
        __syncthreads();
        if (grp == 1) return;
#pragma unroll
        for (int u = 0; u < NT; ++u) acc[u] += sum[u * 64];
        if (bias) bsum += bs[0];
    }
    if (bias) {
        // lanes r, r + 16, r + 32, r + 48 hold row r: fixed pairing order
        const float s1 = bsum + __shfl_xor(bsum, 16);
        const float s2 = s1 + __shfl_xor(s1, 32);
        if (q == 0 && n0 + r < cout) bpart[(int64_t)c * cout + n0 + r] = s2;
    }
    // column r of tile u: its tap's channel
#pragma unroll
    for (int u = 0; u < NT; ++u) {
        const int dx = HALF ? 2 * u + (r >> 3) : u;
        if (dx > 2) continue;
        const int k = ((dzi * 3 + wave) * 3 + dx) * cin + ci0 + (HALF ? r & 7 : r);
#pragma unroll
        for (int j = 0; j < 4; ++j) part[((int64_t)c * coutp + n0 + 4 * q + j) * kp + k] = acc[u][j];
    }
    // the padding columns
    if (first)
        for (int i = tid; i < 16 * (kp - 27 * cin); i += 192) {
            const int pad = kp - 27 * cin, row = i / pad;
            part[((int64_t)c * coutp + n0 + row) * kp + 27 * cin + i - row * pad] = 0.f;
        }
}

// W'[ci][tap' * cout + co] = W[co][(26 - tap') * cin + ci]  (bf16, padded: ci to 16, k' to 32)
struct Flip {
    const __bf16* W;
    int cin, kp, cout, kp2, cinp;
    __bf16* Wt;

    __device__ __forceinline__ void entry(int64_t i) const {
        if (i >= (int64_t)cinp * kp2) return;
        const int ci = (int)(i / kp2), k2 = (int)(i - (int64_t)ci * kp2);
        __bf16 v = (__bf16)0.f;
        if (ci < cin && k2 < 27 * cout) {
            const int tp = k2 / cout, co = k2 - tp * cout;
            v = W[(int64_t)co * kp + (26 - tp) * cin + ci];
        }
        Wt[i] = v;
    }
};

__global__ void k_flip_weights(Flip f) { f.entry((int64_t)blockIdx.x * blockDim.x + threadIdx.x); }

// dW[i] (+)= sum over chunks of part[chunk][i], i < n, and in the blocks after those,
// db[i] (+)= the same over bpart[chunk][i], i < nb (bpart null: no bias).  A block covers
// 32 entries with 8 groups of 32 threads: group g adds chunks g, g + 8, g + 16, ... in order,
// then the 8 group sums are added in group order (a fixed order for every launch).
// The last blocks flip the layer's weights for the data gradient that follows: on the layers of
// a 64^3 training step the sums take 5 us and the flip took 3.5 as a launch of its own, both
// little more than the launch; together they take 5.7.
__global__ __launch_bounds__(256) void k_sum_chunks(const float* __restrict__ part, int nchunk, int64_t n,
                                                    const float* __restrict__ bpart, int nb, int accumulate,
                                                    float* __restrict__ dw, float* __restrict__ db, int64_t sums, Flip flip) {
    if ((int64_t)blockIdx.x >= sums) {
        flip.entry(((int64_t)blockIdx.x - sums) * 256 + threadIdx.x);
        return;
    }
    __shared__ float red[8][32];
    const int x = threadIdx.x & 31, grp = threadIdx.x >> 5;
    const int64_t wblocks = (n + 31) / 32;
    const bool bias = (int64_t)blockIdx.x >= wblocks;
    const float* src = bias ? bpart : part;
    float* dst = bias ? db : dw;
    const int64_t len = bias ? nb : n;
    const int64_t i = ((int64_t)blockIdx.x - (bias ? wblocks : 0)) * 32 + x;
    float s = 0.f;
    if (i < len)
        for (int c = grp; c < nchunk; c += 8) s += src[(int64_t)c * len + i];
    red[grp][x] = s;
    __syncthreads();
    if (grp == 0 && i < len) {
        float t = red[0][x];
#pragma unroll
        for (int g = 1; g < 8; ++g) t += red[g][x];
        dst[i] = accumulate ? dst[i] + t : t;
    }
}

__global__ void k_to_bf16(const float* __restrict__ x, int64_t n, __bf16* __restrict__ y) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = (__bf16)x[i];
}

// Pooling, upsampling and the branch points of the network.  Fine grid D x H x W (even), coarse
// D/2 x H/2 x W/2.  These kernels only move bytes, so each makes its pass once and in whole 16-byte
// accesses: a thread holds V = 8 consecutive channels (V = 1 where a channel count is no multiple
// of 8 or a pointer is not aligned), consecutive threads write consecutive units of a row, and a
// workgroup takes whole rows of its output, so that the row's indices are uniform and the only
// division per unit is that by the units of a voxel.  One value per thread and one kernel per
// operand took 95 us (upsampling) and 38 us (skip channels) where the joint pass takes 23,
// averages over the three scales of a 128^3 prediction with 16, 32, 64, 128 channels.
template <int V>
struct Channels {
    typedef __bf16 vec __attribute__((ext_vector_type(V)));
    vec v;
    __device__ __forceinline__ static Channels load(const __bf16* p, int64_t unit) {
        return {*reinterpret_cast<const vec*>(p + unit * V)};
    }
    __device__ __forceinline__ void store(__bf16* p, int64_t unit) const { *reinterpret_cast<vec*>(p + unit * V) = v; }
};

// How the rows of an output are walked: a workgroup to a row; `segs` workgroups to a row; a
// workgroup to the rows that its threads hold at 1 << lanes threads each.
enum class Rows { WHOLE, CUT, SHARED };
struct RowSplit {
    int segs, lanes;
};

// The D x H rows of the output (and again beyond the launch), their units walked by the threads:
// f(plane, row of the plane, row, voxel x, unit of the voxel).  The row is uniform but for SHARED.
template <Rows MODE, class Fn>
__device__ __forceinline__ void each_row(int D, int H, int W, FastDiv cu, RowSplit sp, Fn&& f) {
    const int n = W * (int)cu.d;
    auto walk = [&](int row, unsigned first, unsigned step) {
        const int z = row / H, y = row - z * H;
        for (unsigned e = first; e < (unsigned)n; e += step) {
            const int x = cu.mul | cu.one ? quot((int)e, cu) : (int)(e / cu.d);
            f(z, y, row, x, (int)(e - x * cu.d));
        }
    };
    if (MODE == Rows::WHOLE) {
        for (int row = blockIdx.x; row < D * H; row += gridDim.x) walk(row, threadIdx.x, blockDim.x);
    } else if (MODE == Rows::CUT) {  // few rows, all of them in the launch
        const int row = blockIdx.x / sp.segs, seg = blockIdx.x - row * sp.segs;
        walk(row, seg * blockDim.x + threadIdx.x, sp.segs * blockDim.x);
    } else {
        const int64_t held = blockDim.x >> sp.lanes;
        for (int64_t row = blockIdx.x * held + (threadIdx.x >> sp.lanes); row < (int64_t)D * H; row += gridDim.x * held)
            walk((int)row, threadIdx.x & ((1u << sp.lanes) - 1), 1u << sp.lanes);
    }
}

// 2x2x2 average pool; C in units
template <int V, Rows MODE>
__global__ __launch_bounds__(256) void k_pool2(const __bf16* __restrict__ x, Grid3 f, FastDiv C, RowSplit sp, __bf16* __restrict__ y) {
    const int Wc = f.W / 2, cu = (int)C.d;
    each_row<MODE>(f.D / 2, f.H / 2, Wc, C, sp, [&](int zc, int yc, int row, int xc, int c) {
        const int64_t fine = ((int64_t)2 * zc * f.H + 2 * yc) * f.W;
        Channels<V> in[8], out;
#pragma unroll
        for (int m = 0; m < 8; ++m)
            in[m] = Channels<V>::load(x, (fine + ((int64_t)(m >> 2) * f.H + (m >> 1 & 1)) * f.W + 2 * xc + (m & 1)) * cu + c);
#pragma unroll
        for (int k = 0; k < V; ++k) {
            float s = 0.f;
#pragma unroll
            for (int m = 0; m < 8; ++m) s += bf2f(in[m].v[k]);
            out.v[k] = (__bf16)(0.125f * s);
        }
        out.store(y, ((int64_t)row * Wc + xc) * cu + c);
    });
}

// Adjoint of the pool (dy coarse -> fine), added to the gradient of the other branch (a, null:
// none; channels [ca0, ca0 + C) of a tensor of Ca) and passed through the ReLU of the layer
// (gate, null: none):  out = (a + dy / 8) [gate > 0].  All channel counts in units.
template <int V, Rows MODE>
__global__ __launch_bounds__(256) void k_pool2_bwd(const __bf16* __restrict__ dy, Grid3 f, FastDiv C, RowSplit sp,
                                                   const __bf16* __restrict__ a, int Ca, int ca0,
                                                   const __bf16* __restrict__ gate, __bf16* __restrict__ out) {
    const int cu = (int)C.d;
    each_row<MODE>(f.D, f.H, f.W, C, sp, [&](int z, int y, int row, int x, int c) {
        const int64_t coarse = ((int64_t)(z / 2) * (f.H / 2) + y / 2) * (f.W / 2), fine = (int64_t)row * f.W;
        const Channels<V> d = Channels<V>::load(dy, (coarse + x / 2) * cu + c);
        Channels<V> va, vg, o;
        if (a) va = Channels<V>::load(a, (fine + x) * Ca + ca0 + c);
        if (gate) vg = Channels<V>::load(gate, (fine + x) * cu + c);
#pragma unroll
        for (int k = 0; k < V; ++k) {
            const __bf16 p = (__bf16)(0.125f * bf2f(d.v[k]));
            __bf16 r = a ? (__bf16)(bf2f(va.v[k]) + bf2f(p)) : p;
            if (gate && !(bf2f(vg.v[k]) > 0.f)) r = (__bf16)0.f;
            o.v[k] = r;
        }
        o.store(out, (fine + x) * cu + c);
    });
}

// Nearest 2x upsampling of `low` (Cl channels) and, beside it, the Cs channels of `skip`, into
// channels [c0, c0 + Cl + Cs) of a fine tensor of Ct; C = Cl + Cs, all in units.
template <int V, Rows MODE>
__global__ __launch_bounds__(256) void k_up2(const __bf16* __restrict__ low, int Cl, const __bf16* __restrict__ skip,
                                             Grid3 f, FastDiv C, RowSplit sp, int Ct, int c0, __bf16* __restrict__ y) {
    const int Cs = (int)C.d - Cl;
    each_row<MODE>(f.D, f.H, f.W, C, sp, [&](int z, int yy, int row, int x, int c) {
        const int64_t coarse = ((int64_t)(z / 2) * (f.H / 2) + yy / 2) * (f.W / 2), fine = (int64_t)row * f.W;
        const bool up = c < Cl;
        const Channels<V> v = Channels<V>::load(up ? low : skip, up ? (coarse + x / 2) * Cl + c : (fine + x) * Cs + c - Cl);
        v.store(y, (fine + x) * Ct + c0 + c);
    });
}

// Adjoint of the upsampling: the sums over 2x2x2 voxels of channels [c0, c0 + C) of a fine tensor
// of Ct, passed through the ReLU of the coarse layer (gate, null: none).  All counts in units.
template <int V, Rows MODE>
__global__ __launch_bounds__(256) void k_up2_bwd(const __bf16* __restrict__ dy, Grid3 f, FastDiv C, RowSplit sp, int Ct, int c0,
                                                 const __bf16* __restrict__ gate, __bf16* __restrict__ dx) {
    const int Wc = f.W / 2, cu = (int)C.d;
    each_row<MODE>(f.D / 2, f.H / 2, Wc, C, sp, [&](int zc, int yc, int row, int xc, int c) {
        const int64_t fine = ((int64_t)2 * zc * f.H + 2 * yc) * f.W;
        const int64_t at = ((int64_t)row * Wc + xc) * cu + c;
        Channels<V> in[8], vg, out;
#pragma unroll
        for (int m = 0; m < 8; ++m)
            in[m] = Channels<V>::load(dy, (fine + ((int64_t)(m >> 2) * f.H + (m >> 1 & 1)) * f.W + 2 * xc + (m & 1)) * Ct + c0 + c);
        if (gate) vg = Channels<V>::load(gate, at);
#pragma unroll
        for (int k = 0; k < V; ++k) {
            float s = 0.f;
#pragma unroll
            for (int m = 0; m < 8; ++m) s += bf2f(in[m].v[k]);
            out.v[k] = (__bf16)s;
            if (gate) out.v[k] = bf2f(vg.v[k]) > 0.f ? (__bf16)(bf2f(out.v[k]) + 0.f) : (__bf16)0.f;
        }
        out.store(dx, at);
    });
}

// copy channels [c0, c0 + C) between a C-channel tensor and a Ct-channel tensor
__global__ void k_channels(const __bf16* __restrict__ src, int64_t nvox, int C, int Ct, int c0, int into_wide,
                           __bf16* __restrict__ dst) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nvox * C) return;
    const int64_t v = i / C;
    const int c = (int)(i % C);
    if (into_wide) dst[v * Ct + c0 + c] = src[i];
    else dst[i] = src[v * Ct + c0 + c];
}

// out = (a + b) * [gate > 0]  (b and gate optional): gradients meeting at a branch point and
// the ReLU derivative
__global__ void k_add_gate(const __bf16* __restrict__ a, const __bf16* __restrict__ b, const __bf16* __restrict__ gate,
                           int64_t n, __bf16* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float v = bf2f(a[i]) + (b ? bf2f(b[i]) : 0.f);
    if (gate && !(bf2f(gate[i]) > 0.f)) v = 0.f;
    out[i] = (__bf16)v;
}

// masked mean-squared error over the first `cout` channels: loss partials per block and
// dY = 2 (y - t) mask / count as bf16
__global__ __launch_bounds__(256) void k_mse(const float* __restrict__ y, const float* __restrict__ t,
                                             const float* __restrict__ mask, int64_t M, int cout, float inv_count,
                                             __bf16* __restrict__ dy, double* __restrict__ part) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    double e = 0.0;
    if (i < M * cout) {
        const float w = mask[i / cout];
        const float d = (y[i] - t[i]) * w;
        e = (double)d * d;
        dy[i] = (__bf16)(2.f * d * inv_count);
    }
    __shared__ double red[256];
    red[threadIdx.x] = e;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// Adam step on fp32 master weights; refreshes the bf16 copies.  One launch for up to ADAM_MAX
// tensors, the launch's blocks split between them in order (first[t]: the first block of tensor
// t): a network's weights are many small tensors, and a launch apiece took 24 x 2.2 us of a 64^3
// training step, one takes 9.7.
constexpr int ADAM_MAX = 48;  // at most a wave's lanes, and 4 KiB of kernel arguments
struct AdamList {
    mfnn_adam_tensor t[ADAM_MAX];
    uint32_t first[ADAM_MAX];
    int count;
};

// Value i of a tensor: all loads before the stores.
__device__ __forceinline__ void adam_value(int64_t i, float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m1,
                                           float* __restrict__ m2, __bf16* __restrict__ wb, float lr, float b1, float b2,
                                           float eps, float c1, float c2) {
    const float gi = g[i], wi = w[i];
    const float a = b1 * m1[i] + (1.f - b1) * gi;
    const float b = b2 * m2[i] + (1.f - b2) * gi * gi;
    m1[i] = a;
    m2[i] = b;
    const float v = wi - lr * (a * c1) / (sqrtf(b * c2) + eps);
    w[i] = v;
    if (wb) wb[i] = (__bf16)v;
}

__global__ __launch_bounds__(256) void k_adam_many(AdamList list, float lr, float b1, float b2, float eps, float c1, float c2) {
    const int lane = threadIdx.x & 63;
    const int k = __builtin_amdgcn_readfirstlane(
        (int)__popcll(__ballot(lane < list.count && blockIdx.x >= list.first[lane < ADAM_MAX ? lane : 0])) - 1);
    const mfnn_adam_tensor& t = list.t[k];
    const int64_t i = (int64_t)(blockIdx.x - list.first[k]) * 256 + threadIdx.x;
    if (i < t.n) adam_value(i, t.w, t.g, t.m1, t.m2, static_cast<__bf16*>(t.wb), lr, b1, b2, eps, c1, c2);
}

// A tensor alone: no lookup, and a tenth of the arguments (us, in a list of one and so: 30 M values
// 180 and 149, 1000 values 7.1 and 5.4).
__global__ __launch_bounds__(256) void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m1,
                                              float* __restrict__ m2, int64_t n, float lr, float b1, float b2, float eps,
                                              float c1, float c2, __bf16* __restrict__ wb) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) adam_value(i, w, g, m1, m2, wb, lr, b1, b2, eps, c1, c2);
}

inline unsigned nblk(int64_t n, int b = 256) { return (unsigned)((n + b - 1) / b); }

template <class... P>
inline bool aligned16(P... p) {
    return (((uintptr_t)p | ...) & 15) == 0;
}

// Launch of a kernel that takes its D x H x W output in rows (each_row), C channels in units of 8
// (wide) or 1: launch(channels per unit, mode, workgroups, threads, units of a voxel, split).  A
// workgroup to a row fills the chip where rows are many and long enough; else few long rows are cut
// until 512 workgroups have a share (at least a unit to each thread), and many rows shorter than a
// wave share workgroups (us a pass, a workgroup to a row and so: up of 24 channels on 2 x 6 x 1380 29.4
// and 4.7, of 3 channels on 194 x 206 x 2 10.9 and 4.7, a launch each).  A division of a row's unit by the units
// of a voxel is exact below 2^32 (FastDiv), else left to the kernel.
constexpr int MAX_ROW_GROUPS = 1 << 24;  // a launch holds fewer than 2^32 threads
template <class Fn>
int rows_of(int64_t D, int64_t H, int64_t W, int C, bool wide, Fn&& launch) {
    const int64_t rows = D * H, cu = wide ? C / 8 : C, n = W * cu;
    if (rows <= 0 || n <= 0) return -2;
    if (rows > INT32_MAX - MAX_ROW_GROUPS || n > INT32_MAX - 256) return -1;
    FastDiv c = fast_div((uint32_t)cu);
    if (n * cu >= (int64_t)1 << 32) c.mul = c.one = 0;
    RowSplit sp{1, 0};
    auto with = [&](auto mode, int64_t groups, int threads) {
        const int g = (int)std::min<int64_t>(groups, MAX_ROW_GROUPS);
        if (wide) launch(std::integral_constant<int, 8>{}, mode, g, threads, c, sp);
        else launch(std::integral_constant<int, 1>{}, mode, g, threads, c, sp);
    };
    if (n <= 64 && rows > 4096) {
        while ((1 << sp.lanes) < n) ++sp.lanes;
        const int64_t held = 256 >> sp.lanes;
        with(std::integral_constant<Rows, Rows::SHARED>{}, (rows + held - 1) / held, 256);
    } else if (rows < 512 && n > 256) {
        sp.segs = (int)std::min<int64_t>((511 + rows) / rows, (n + 255) / 256);
        with(std::integral_constant<Rows, Rows::CUT>{}, rows * sp.segs, 256);
    } else {
        with(std::integral_constant<Rows, Rows::WHOLE>{}, rows, (int)std::min<int64_t>(256, (n + 63) / 64 * 64));
    }
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int conv_launch(const __bf16* X, const __bf16* Wb, const float* bias, const __bf16* gate, const Grid3& g, int cin, int kp,
                int cout, int relu, __bf16* yb, float* yf, hipStream_t s) {
    const int ntw = (cout + 15) / 16;
    const bool quad = cout % 4 == 0 && (uintptr_t)bias % 16 == 0 && (uintptr_t)gate % 8 == 0 && (uintptr_t)yb % 8 == 0 &&
                     (uintptr_t)yf % 16 == 0;
    const Epilogue ep{bias, gate, yb, yf, cout, relu, quad};
    const ConvPlan* const plan = kept_plan(g, cin, ntw);
    if (!plan) {
        const int64_t M = (int64_t)g.D * g.H * g.W;
        // grids of 65536 voxels and more with one or two channel tiles: two voxel tiles per wave, but not
        // one channel tile of deep inputs beyond the caches (us, one voxel tile and two: 128^3 48 -> 16
        // 615 and 530, 448 -> 32 15900 and 10850, 48^3 1104 -> 16 1390 and 1113; 64^3 1104 -> 16 3195 and
        // 4100)
        const bool pair = M >= 65536 && !(ntw == 1 && cin > 512 && M >= 1 << 18);
        switch (gather_single(g, ntw) ? 0 : ntw) {
#define MFNN_GATHER(n, m) k_conv3<n, m><<<dim3(nblk(M, 64 * m), (ntw + n - 1) / n), 256, 0, s>>>(X, Wb, g, cin, kp, ntw, ep)
            case 0: MFNN_GATHER(1, 1); break;
            case 1: if (pair) MFNN_GATHER(1, 2); else MFNN_GATHER(1, 1); break;
            case 2: if (pair) MFNN_GATHER(2, 2); else MFNN_GATHER(2, 1); break;
            case 3: MFNN_GATHER(3, 1); break;
            case 4: MFNN_GATHER(4, 1); break;
            case 5: MFNN_GATHER(5, 1); break;
            case 6: MFNN_GATHER(6, 1); break;
            case 7: MFNN_GATHER(7, 1); break;
            case 8: MFNN_GATHER(8, 1); break;
            default: MFNN_GATHER(12, 1); break;
#undef MFNN_GATHER
        }
        return hipGetLastError() == hipSuccess ? 0 : -2;
    }
    const ConvPlan& p = *plan;
    const dim3 grid(p.boxes, (ntw + p.nt - 1) / p.nt);
    switch (10 * p.mt + p.nt) {
#define MFNN_BOX(m, n, pf) \
    case 10 * m + n: k_conv3_box<m, n, pf><<<grid, 256, p.lds, s>>>(X, Wb, g, cin, kp, ntw, ep, p.t); break;
        MFNN_BOX(1, 1, 8) MFNN_BOX(1, 2, 4) MFNN_BOX(1, 3, 4) MFNN_BOX(1, 4, 4)
        MFNN_BOX(2, 1, 4) MFNN_BOX(2, 2, 4) MFNN_BOX(2, 3, 2) MFNN_BOX(2, 4, 2)
        MFNN_BOX(4, 1, 4) MFNN_BOX(4, 2, 2) MFNN_BOX(4, 3, 2)
        MFNN_BOX(8, 1, 2) MFNN_BOX(8, 2, 2)
#undef MFNN_BOX
    }
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace

extern "C" {

void* mfnn_alloc(int64_t bytes) {
    std::lock_guard<std::recursive_mutex> lock(mflbm::device_lock());
    void* p = nullptr;
    if (bytes <= 0 || hipMalloc(&p, (size_t)bytes) != hipSuccess) return nullptr;
    return p;
}

int mfnn_free(void* p) {
    std::lock_guard<std::recursive_mutex> lock(mflbm::device_lock());
    return hipFree(p) == hipSuccess ? 0 : -2;
}

int mfnn_copy(void* dst, const void* src, int64_t bytes, int32_t kind) {
    const hipMemcpyKind k = kind == 0 ? hipMemcpyHostToDevice : (kind == 1 ? hipMemcpyDeviceToHost : hipMemcpyDeviceToDevice);
    if (bytes < 0 || kind < 0 || kind > 2) return -1;
    return hipMemcpy(dst, src, (size_t)bytes, k) == hipSuccess ? 0 : -2;
}

int mfnn_zero(void* dst, int64_t bytes) {
    if (bytes < 0) return -1;
    return hipMemset(dst, 0, (size_t)bytes) == hipSuccess ? 0 : -2;
}

int mfnn_sync(void) { return hipDeviceSynchronize() == hipSuccess ? 0 : -2; }

int mfnn_conv3(const void* x, const void* w, const float* bias, const void* gate, int32_t D, int32_t H, int32_t W,
               int32_t cin, int32_t kp, int32_t cout, int32_t relu, void* yb, float* yf, void* stream) {
    if (cin % 8 || kp % 32 || kp < 27 * cin || cout <= 0 || cout > 192 || D <= 0 || H <= 0 || W <= 0) return -1;
    if ((uintptr_t)x % 16 || (uintptr_t)w % 16) return -1;  // 16-byte operand loads
    return conv_launch((const __bf16*)x, (const __bf16*)w, bias, (const __bf16*)gate, Grid3{D, H, W}, cin, kp, cout, relu,
                       (__bf16*)yb, yf, (hipStream_t)stream);
}

int64_t mfnn_wgrad_workspace(int32_t D, int32_t H, int32_t W, int32_t kp, int32_t cout, int32_t chunk) {
    const int64_t M = (int64_t)D * H * W;
    const int64_t nchunk = (M + chunk - 1) / chunk;
    return nchunk * ((int64_t)((cout + 15) / 16 * 16) * kp + cout);  // weight partials, then bias partials
}

}  // extern "C"

namespace {

bool wgrad_args_ok(const void* x, const void* dz, int32_t D, int32_t H, int32_t W, int32_t cin, int32_t kp,
                   int32_t cout, int32_t chunk) {
    if (cin % 8 || cout % 8 || cin <= 0 || cout <= 0 || kp % 32 || kp < 27 * cin || chunk <= 0 || chunk % 32) return false;
    if (D <= 0 || H <= 0 || W <= 0) return false;
    return (uintptr_t)x % 16 == 0 && (uintptr_t)dz % 16 == 0;  // 16-byte operand loads
}

// Waves of k_conv3_wgrad with one tile each.
inline int64_t wgrad_waves(int kp, int coutp, int nchunk) { return (int64_t)(kp / 16) * (coutp / 16) * nchunk; }

// Whether the rows kernel is the faster one.  It loads at least three rows for the voxels that it
// stages, and LDS holds fewer voxels of wider rows (512 of 90, 256 of 200, 128 beyond), so that wide
// grids lose on it, the sooner the fewer voxels share its start: us of 12 x 12 rows 32 -> 32, with it
// and with k_conv3_wgrad, 204 wide 21 and 25, 280 32.1 and 31.8, 360 44 and 34; of 8 x 64 rows 340 wide
// 0.93 of the time, 360 1.19; of 16 x 200 rows 360 wide level.  Inputs of one slice of channels keep
// it longer.  A count of channels with 8 over takes it two launches: 24 -> 24 on 165 voxels 11 and 7.5,
// 72 -> 128 on 2544 18.7 and 24.5.  On fewer than 128 voxels its 16-channel slices are the longer chain:
// 192 -> 40 on 6 voxels 8.8 and 7.1.
bool rows_pay(const Grid3& g, int cin, int waves) {
    const int64_t M = (int64_t)g.D * g.H * g.W;
    const bool two = cin > 16 && cin % 16;  // launches
    if (M < 128 && waves >= 500) return false;
    if (two && waves < (g.W >= 128 ? 2000 : 1200)) return false;
    if (cin == 8) return M < 65536 || g.W <= 512;
    if (M < 65536) return g.W <= (two ? 212 : cin == 16 ? 340 : 270);
    return M >= 1 << 19 || cin == 16 || g.W <= (two ? 230 : 340);
}

// Launches k_conv3_wgrad_rows over all chunks; false where its rows do not fit LDS or do not pay.
bool wgrad_rows(const __bf16* X, const __bf16* dZ, const Grid3& g, int cin, int kp, int coutp, int cout, int chunk,
                int nchunk, float* part, float* bpart, hipStream_t s) {
    if (!rows_pay(g, cin, (int)std::min<int64_t>(wgrad_waves(kp, coutp, nchunk), 1 << 20))) return false;
    const int full = cin / 16, ntiles = coutp / 16;
    auto launch = [&](bool half) {
        const int64_t vb = half ? 16 : 32, WP = g.W + 2, WH = (int64_t)g.W * g.H;
        WgradRows t;
        t.ci0 = half ? 16 * full : 0;
        // as many voxels at a time as 48 KB hold (three workgroups per CU); wide rows take more
        // LDS, down to 128 voxels at a time
        int64_t lds = 0;
        for (t.sub = 512;; t.sub /= 2) {
            const int64_t rows = (t.sub + g.W - 2) / g.W + 2 * ((t.sub + WH - 2) / WH) + 3;
            t.lds_dz = (int)(128 + std::min<int64_t>(rows * WP * vb, 1 << 20));
            t.lds_pos = t.lds_dz + t.sub * 32;
            lds = std::max<int64_t>(t.lds_pos + 4 * t.sub, 3 * 64 * 3 * 16 + 64 * 4);  // and the second group's sums
            if (lds <= 48 * 1024 || t.sub == 128) break;
        }
        t.gx = 3 * (half ? 1 : full);
        t.gy = ntiles;
        const int64_t M = WH * g.D, wgs = (int64_t)t.gx * t.gy * nchunk;
        // exact quotients; 24-bit products and 31-bit offsets of the loads; threads of the launch
        if (lds > 80 * 1024 || (int64_t)(g.H + 2) * (g.H + 600) >= (1ll << 32) || (int64_t)(g.W + 600) * g.W >= (1ll << 32) ||
            (int64_t)g.D * g.H >= (1 << 24) || 2ll * g.W * cin >= (1 << 24) || 2 * M * std::max(cin, cout) >= NOWHERE ||
            wgs >= 1 << 23)
            return false;
        // The workgroups of a chunk read the same rows and the same dZ.  On inputs that an XCD's
        // 4 MB L2 holds a good part of, they may lie anywhere; beyond, they go to one XCD (us, in
        // turn and contiguous: 16^3 192 -> 64 22.1 and 23.7, 32^3 96 -> 32 31.9 and 32.8, 64^3
        // 16 -> 16 29.1 and 29.0, 48 -> 16 59.3 and 48.3, 128^3 48 -> 16 528 and 323).
        t.per_xcd = 2 * M * (cin + cout) > 16 << 20;
        // Up to two workgroups per CU the staging and the operand latency bound a workgroup, and a
        // second group of waves halves both (us with one and two: 64^3 16 -> 16 29.1 and 25.2, 16^3
        // 32 -> 64 9.3 and 8.4); beyond, more workgroups per CU do better (32^3 32 -> 32 16.0 and
        // 16.9, 128^3 16 -> 16 142 and 183).
        const bool two = wgs <= 512;
        t.planes = WH >= t.sub && chunk > t.sub;
        t.row = fast_div((uint32_t)(WP * vb / 16));
        t.h2 = fast_div(g.H + 2);
        t.w = fast_div(g.W);
        t.h = fast_div(g.H);
#define MFNN_ROWS(h, gr) \
    k_conv3_wgrad_rows<h, gr><<<(unsigned)wgs, 192 * gr, lds, s>>>(X, dZ, g, cin, kp, coutp, cout, chunk, t, part, bpart)
        if (half) {
            if (two) MFNN_ROWS(true, 2);
            else MFNN_ROWS(true, 1);
        } else {
            if (two) MFNN_ROWS(false, 2);
            else MFNN_ROWS(false, 1);
        }
#undef MFNN_ROWS
        return true;
    };
    if (full && !launch(false)) return false;
    return cin % 16 == 0 || launch(true);
}

bool flip_args_ok(int32_t cin, int32_t cout, int32_t kp2, int32_t cinp) {
    return kp2 >= 27 * cout && kp2 % 32 == 0 && cinp >= cin && cinp % 16 == 0;
}

// The weight-gradient launches of valid arguments: partials into `work`, then the chunk sums and,
// with flip.Wt, the flipped weights.
int wgrad_launch(const void* x, const void* dz, int32_t D, int32_t H, int32_t W, int32_t cin, int32_t kp, int32_t cout,
                 int32_t chunk, float* work, float* dw, float* db, int32_t accumulate, const Flip& flip, void* stream) {
    const Grid3 g{D, H, W};
    const int64_t M = (int64_t)D * H * W;
    const int nchunk = (int)((M + chunk - 1) / chunk);
    const int coutp = (cout + 15) / 16 * 16;
    hipStream_t s = (hipStream_t)stream;
    const int64_t n = (int64_t)coutp * kp;
    float* bpart = db ? work + nchunk * n : nullptr;
    const __bf16 *X = (const __bf16*)x, *dZ = (const __bf16*)dz;
    if (!wgrad_rows(X, dZ, g, cin, kp, coutp, cout, chunk, nchunk, work, bpart, s)) {
        // Two k tiles per wave halve the dZ loads, one keeps twice the waves: the second wins where the
        // grid of single tiles has fewer than 3072 waves (three per SIMD) and on up to 16 channels on both
        // sides (us, one and two: 8 x 64 x 512 16 -> 16 75 and 87, 48 -> 16 200 and 131, 1 x 38 x 623 16
        // -> 144 42 and 36, 256^3 64 -> 64 58300 and 46300).  kp is a multiple of 32.
        if (std::max(cin, cout) > 16 && wgrad_waves(kp, coutp, nchunk) >= 3072)
            k_conv3_wgrad<2><<<dim3(kp / 32, coutp / 16, nchunk), 64, 0, s>>>(X, dZ, g, cin, kp, coutp, cout, chunk, work, bpart);
        else
            k_conv3_wgrad<1><<<dim3(kp / 16, coutp / 16, nchunk), 64, 0, s>>>(X, dZ, g, cin, kp, coutp, cout, chunk, work, bpart);
    }
    const unsigned sblocks = nblk(n, 32) + (db ? nblk(cout, 32) : 0);
    const unsigned fblocks = flip.Wt ? nblk((int64_t)flip.cinp * flip.kp2) : 0;
    k_sum_chunks<<<sblocks + fblocks, 256, 0, s>>>(work, nchunk, n, bpart, db ? cout : 0, accumulate, dw, db, sblocks, flip);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

// Scratch of mfnn_conv3_wgrad_static: every partial it sums is written first by the
// partial kernels of the same call, so no call needs it cleared.  In host code `scratch`
// names a host-side shadow, not the device array: the device address comes from
// hipGetSymbolAddress, once per device (each device holds its own copy of the array).
static __device__ __align__(256) float scratch[MFNN_WGRAD_SCRATCH_FLOATS];
constexpr int MAX_DEVICES = 64;
std::mutex scratch_mutex;
float* scratch_dev[MAX_DEVICES] = {};

// Address of the current device's scratch (null on a runtime error).
float* scratch_address() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return nullptr;
    std::lock_guard<std::mutex> lock(scratch_mutex);
    if (!scratch_dev[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
        scratch_dev[dev] = static_cast<float*>(p);
    }
    return scratch_dev[dev];
}

}  // namespace

extern "C" {

int mfnn_conv3_wgrad(const void* x, const void* dz, int32_t D, int32_t H, int32_t W, int32_t cin, int32_t kp,
                     int32_t cout, int32_t chunk, float* work, float* dw, float* db, int32_t accumulate, void* stream) {
    if (!wgrad_args_ok(x, dz, D, H, W, cin, kp, cout, chunk)) return -1;
    return wgrad_launch(x, dz, D, H, W, cin, kp, cout, chunk, work, dw, db, accumulate, Flip{}, stream);
}

int mfnn_conv3_wgrad_static(const void* x, const void* dz, int32_t D, int32_t H, int32_t W, int32_t cin, int32_t kp,
                            int32_t cout, int32_t chunk, float* dw, float* db, int32_t accumulate, void* stream) {
    if (!wgrad_args_ok(x, dz, D, H, W, cin, kp, cout, chunk)) return -1;
    if (mfnn_wgrad_workspace(D, H, W, kp, cout, chunk) > (int64_t)MFNN_WGRAD_SCRATCH_FLOATS) return -3;
    float* work = scratch_address();
    if (!work) return -2;
    return wgrad_launch(x, dz, D, H, W, cin, kp, cout, chunk, work, dw, db, accumulate, Flip{}, stream);
}

int mfnn_conv3_wgrad_flip(const void* x, const void* dz, int32_t D, int32_t H, int32_t W, int32_t cin, int32_t kp,
                          int32_t cout, int32_t chunk, float* work, float* dw, float* db, int32_t accumulate, const void* w,
                          int32_t kp2, int32_t cinp, void* wt, void* stream) {
    if (!wgrad_args_ok(x, dz, D, H, W, cin, kp, cout, chunk) || !flip_args_ok(cin, cout, kp2, cinp) || !w || !wt) return -1;
    return wgrad_launch(x, dz, D, H, W, cin, kp, cout, chunk, work, dw, db, accumulate,
                        Flip{(const __bf16*)w, cin, kp, cout, kp2, cinp, (__bf16*)wt}, stream);
}

int mfnn_flip_weights(const void* w, int32_t cin, int32_t kp, int32_t cout, int32_t kp2, int32_t cinp, void* wt,
                      void* stream) {
    if (!flip_args_ok(cin, cout, kp2, cinp)) return -1;
    const int64_t n = (int64_t)cinp * kp2;
    k_flip_weights<<<nblk(n), 256, 0, (hipStream_t)stream>>>(Flip{(const __bf16*)w, cin, kp, cout, kp2, cinp, (__bf16*)wt});
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int mfnn_to_bf16(const float* x, int64_t n, void* y, void* stream) {
    k_to_bf16<<<nblk(n), 256, 0, (hipStream_t)stream>>>(x, n, (__bf16*)y);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int mfnn_pool2(const void* x, int32_t D, int32_t H, int32_t W, int32_t C, void* y, int32_t backward, void* stream) {
    if (backward) return mfnn_pool2_merge(x, D, H, W, C, nullptr, C, 0, nullptr, y, stream);
    if (D % 2 || H % 2 || W % 2) return -1;
    const Grid3 f{D, H, W};
    hipStream_t s = (hipStream_t)stream;
    return rows_of(D / 2, H / 2, W / 2, C, C % 8 == 0 && aligned16(x, y), [&](auto V, auto mode, int groups, int threads, FastDiv c, RowSplit sp) {
        k_pool2<V, mode><<<groups, threads, 0, s>>>((const __bf16*)x, f, c, sp, (__bf16*)y);
    });
}

int mfnn_pool2_merge(const void* dy, int32_t D, int32_t H, int32_t W, int32_t C, const void* a, int32_t ca, int32_t ca0,
                     const void* gate, void* out, void* stream) {
    if (D % 2 || H % 2 || W % 2 || ca0 < 0 || ca0 + C > ca) return -1;
    const Grid3 f{D, H, W};
    hipStream_t s = (hipStream_t)stream;
    const bool wide = C % 8 == 0 && ca % 8 == 0 && ca0 % 8 == 0 && aligned16(dy, a, gate, out);
    return rows_of(D, H, W, C, wide, [&](auto V, auto mode, int groups, int threads, FastDiv c, RowSplit sp) {
        k_pool2_bwd<V, mode><<<groups, threads, 0, s>>>((const __bf16*)dy, f, c, sp, (const __bf16*)a, ca / V, ca0 / V,
                                                (const __bf16*)gate, (__bf16*)out);
    });
}

int mfnn_up2(const void* x, int32_t D, int32_t H, int32_t W, int32_t C, int32_t ct, int32_t c0, void* y,
             int32_t backward, void* stream) {
    if (backward) return mfnn_up2_split(x, D, H, W, C, ct, c0, nullptr, y, stream);
    return mfnn_up2_cat(x, C, nullptr, 0, D, H, W, ct, c0, y, stream);
}

int mfnn_up2_cat(const void* low, int32_t cl, const void* skip, int32_t cs, int32_t D, int32_t H, int32_t W, int32_t ct,
                 int32_t c0, void* y, void* stream) {
    if (D % 2 || H % 2 || W % 2 || cl < 0 || cs < 0 || c0 < 0 || c0 + cl + cs > ct) return -1;
    const Grid3 f{D, H, W};
    hipStream_t s = (hipStream_t)stream;
    const bool wide = cl % 8 == 0 && cs % 8 == 0 && ct % 8 == 0 && c0 % 8 == 0 && aligned16(low, skip, y);
    return rows_of(D, H, W, cl + cs, wide, [&](auto V, auto mode, int groups, int threads, FastDiv c, RowSplit sp) {
        k_up2<V, mode><<<groups, threads, 0, s>>>((const __bf16*)low, cl / V, (const __bf16*)skip, f, c, sp, ct / V, c0 / V, (__bf16*)y);
    });
}

int mfnn_up2_split(const void* dy, int32_t D, int32_t H, int32_t W, int32_t C, int32_t ct, int32_t c0, const void* gate,
                   void* dx, void* stream) {
    if (D % 2 || H % 2 || W % 2 || c0 < 0 || c0 + C > ct) return -1;
    const Grid3 f{D, H, W};
    hipStream_t s = (hipStream_t)stream;
    const bool wide = C % 8 == 0 && ct % 8 == 0 && c0 % 8 == 0 && aligned16(dy, gate, dx);
    return rows_of(D / 2, H / 2, W / 2, C, wide, [&](auto V, auto mode, int groups, int threads, FastDiv c, RowSplit sp) {
        k_up2_bwd<V, mode><<<groups, threads, 0, s>>>((const __bf16*)dy, f, c, sp, ct / V, c0 / V, (const __bf16*)gate, (__bf16*)dx);
    });
}

int mfnn_channels(const void* src, int64_t nvox, int32_t C, int32_t ct, int32_t c0, int32_t into_wide, void* dst,
                  void* stream) {
    if (c0 < 0 || c0 + C > ct) return -1;
    k_channels<<<nblk(nvox * C), 256, 0, (hipStream_t)stream>>>((const __bf16*)src, nvox, C, ct, c0, into_wide,
                                                              (__bf16*)dst);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int mfnn_add_gate(const void* a, const void* b, const void* gate, int64_t n, void* out, void* stream) {
    k_add_gate<<<nblk(n), 256, 0, (hipStream_t)stream>>>((const __bf16*)a, (const __bf16*)b, (const __bf16*)gate, n,
                                                        (__bf16*)out);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int64_t mfnn_mse_partials(int64_t M, int32_t cout) { return (M * cout + 255) / 256; }

int mfnn_mse(const float* y, const float* t, const float* mask, int64_t M, int32_t cout, float inv_count, void* dy,
             double* part, void* stream) {
    k_mse<<<nblk(M * cout), 256, 0, (hipStream_t)stream>>>(y, t, mask, M, cout, inv_count, (__bf16*)dy, part);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int mfnn_adam_many(const mfnn_adam_tensor* list, int32_t count, float lr, float b1, float b2, float eps, int32_t step,
                   void* stream) {
    if (step < 1 || count < 0 || (count && !list)) return -1;
    for (int t = 0; t < count; ++t)
        if (list[t].n < 0) return -1;
    const float c1 = 1.f / (1.f - powf(b1, (float)step));
    const float c2 = 1.f / (1.f - powf(b2, (float)step));
    for (int at = 0; at < count;) {
        AdamList l;
        int64_t blocks = 0;
        for (l.count = 0; l.count < ADAM_MAX && at < count; ++l.count, ++at) {
            const int64_t b = (list[at].n + 255) / 256;
            if (l.count && blocks + b > 1 << 23) break;  // a launch holds fewer than 2^32 threads
            l.t[l.count] = list[at];
            l.first[l.count] = (uint32_t)blocks;
            blocks += b;
        }
        if (!blocks) continue;
        if (l.count == 1)
            k_adam<<<(unsigned)blocks, 256, 0, (hipStream_t)stream>>>(l.t[0].w, l.t[0].g, l.t[0].m1, l.t[0].m2, l.t[0].n, lr, b1,
                                                                      b2, eps, c1, c2, (__bf16*)l.t[0].wb);
        else
            k_adam_many<<<(unsigned)blocks, 256, 0, (hipStream_t)stream>>>(l, lr, b1, b2, eps, c1, c2);
        if (hipGetLastError() != hipSuccess) return -2;
    }
    return 0;
}

int mfnn_adam(float* w, const float* g, float* m1, float* m2, int64_t n, float lr, float b1, float b2, float eps,
              int32_t step, void* wb, void* stream) {
    if (n <= 0) return step < 1 ? -1 : -2;
    const mfnn_adam_tensor t{w, g, m1, m2, n, wb};
    return mfnn_adam_many(&t, 1, lr, b1, b2, eps, step, stream);
}

}  // extern "C"
