// gemm_slab.hip — projections of many rows: y[M, N] = x[M, K] W[N, K]^T in bfloat16 with float32 sums, tiles of 256 W rows by 128 to 256 x rows
// (slab_rows) on the slab loop of chronos_slab.h.  A workgroup per CU walks its tiles; the slab pipeline runs on from one tile into the next, and where the
// last round would leave half of the CUs idle its tiles are halved.  Config 88 of the projection family (gemm_lg.hip has SwiGLU's split-K).
//
// Epilogues, through 4 KiB of LDS per wave so that every store is 16 bytes of a whole line: plain; activation (squared ReLU, GELU); gated
// units over W = [gate; up], of Llama (SwiGLU, roundings of the unfused form kept) and of the hybrid decoders (clamped, any slope and shift);
// the new residual stream with its RMSNorm partials.  NORMP: the folded input RMSNorm as a scale per row.
//
// Bound by the matrix cores (a slab is 2048 of their cycles and takes 2200) and by the last round of tiles.
// Split-K (plain, resid): the tiles are walked once per slice of K and leave float32 slices [S, M, N], whose stores run beside the next
// tile's first slabs where there is one; a second launch sums them in slice order, with the residual and its partials.  For products whose
// tiles are too few for the chip: the tiles of a launch have to fit one round.  us, the residual form's best tiles before -> this: 4096 x
// 14336 at 128 rows 42 -> 36 (16 slices), 256 56 -> 45 (8), 512 76 -> 65 (4), 768 110 -> 86, 1024 119 -> 101 (88 and 13: the slices are 67 MB,
// written and read), 1536 185 -> 147 (2), 2048 198 -> 182; 2560 249 -> 274, not taken.
// One workgroup per tile -> this, us: 8192 x 3648 x 2048 95.8 -> 93.0; 8192 x 6144 x 2048 157 -> 146 (3 rounds); 8192 x 2560 x 1024 (1.25
// rounds) 52 -> 43; 8192 x 4096 x 4096 190 -> 179; a Llama-3 8B prefill of 5952 tokens, four layers, whole 8604 -> 7986.
#include "chronos_act.h"
#include "chronos_gemm.h"
#include "chronos_hip.h"
#include "chronos_slab.h"

namespace chronos {
namespace {

// sum over the 16 lanes of a DPP row, in every lane
__device__ __forceinline__ float row_sum16(float v) {
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xf, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x124, 0xf, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x122, 0xf, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x121, 0xf, 0xf, false));
    return v;
}

template <int MODE, bool NORMP, int NMX>
__global__ void __launch_bounds__(256, 1) gemm_slab_kernel(PPArgs a) {
    constexpr int TR = 32 * NMX;   // x rows of a tile
    constexpr bool PAIR = MODE == kPPSwiglu || MODE == kPPGlu;
    constexpr int OC = PAIR ? 64 : 128, RBY = 2 * OC, NCH = RBY / 16, RPS = 64 / NCH, NK = 16 / RPS;   // a wave's columns, bytes and
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];                            // pieces per row; rows per store
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wn = wave >> 1, wm = wave & 1, in = lane >> 3, piece = ((lane & 7) ^ in) * 8;
    const int nt = PAIR ? a.F / 128 : (a.N + 255) / 256, S = MODE == kPPPart ? a.splitk : 1;
    const int tail = NMX == 8 ? slab_tail(a.M, nt, S) : 0, mt = tail > 0 ? a.M / TR : (a.M + TR - 1) / TR;
    // tiles in groups of gm along x, so that what an XCD runs at a time shares rows of both operands in its L2
    // (kPPPart: slice by slice; the short last rows of all slices behind)
    auto where = [&](int tile, int& tm, int& tn, int& sl) {
        sl = 0;
        if (tail > 0 && tile >= mt * nt * S) {
            tm = mt;
            tn = tile - mt * nt * S;
            if constexpr (MODE == kPPPart) {
                sl = tn / nt;
                tn -= sl * nt;
            }
            return;
        }
        if constexpr (MODE == kPPPart) {
            sl = tile / (mt * nt);
            tile -= sl * mt * nt;
        }
        if (a.gm > 0 && mt > a.gm) {
            const int per = a.gm * nt, grp = tile / per, r = tile - grp * per, gsz = min(a.gm, mt - grp * a.gm);
            tm = grp * a.gm + r % gsz;
            tn = r / gsz;
        } else {
            tm = tile % mt;
            tn = tile / mt;
        }
    };
    auto off = [&](auto NMC, int tile, int m, uint32_t (&wv)[8], auto& xv, const void*& wb) {
        constexpr int NM = decltype(NMC)::value;
        int tm, tn, sl;
        where(tile, tm, tn, sl);
        const int at = MODE == kPPPart ? sl * a.kts * 64 + piece : piece;
        wb = a.w;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int r = 64 * wave + 8 * i + in;
            const int row = !PAIR ? tn * 256 + r : wave < 2 ? tn * 128 + r : a.F + tn * 128 + r - 128;
            wv[i] = ((uint32_t)row * (uint32_t)a.K + at) * 2;
        }
#pragma unroll
        for (int i = 0; i < NM; ++i) xv[i] = ((uint32_t)(tm * TR + m + 8 * (NM * wave + i) + in) * (uint32_t)a.K + at) * 2;
    };
    // NORMP: a lane sums its row's partials; two buffers in turn (a tile's slabs, with their barriers, lie between a buffer's
    // writers and its readers, and between those and the next writers)
    float* inv = reinterpret_cast<float*>(smem + kSlabLds) + 256;
    auto scales = [&](auto NMC, int tile, int m) {
        if constexpr (NORMP) {
            constexpr int RPW = 8 * decltype(NMC)::value;   // rows per wave
            int tm, tn, sl;
            where(tile, tm, tn, sl);
            const int row = RPW * wave + lane % RPW;
            const float* p = a.part_in + (int64_t)min(tm * TR + m + row, a.M - 1) * a.nparts_in;
            f32x4 t = {0.f, 0.f, 0.f, 0.f};
            int i = 0;
            if ((a.nparts_in & 3) == 0) {
#pragma unroll 1
                for (; i + 32 <= a.nparts_in; i += 32) {
                    f32x4 q[8];
#pragma unroll
                    for (int k = 0; k < 8; ++k) q[k] = *reinterpret_cast<const f32x4*>(p + i + 4 * k);
                    t += ((q[0] + q[1]) + (q[2] + q[3])) + ((q[4] + q[5]) + (q[6] + q[7]));
                }
            }
            float ss = (t[0] + t[1]) + (t[2] + t[3]);
#pragma unroll 1
            for (; i < a.nparts_in; ++i) ss += p[i];
            inv = reinterpret_cast<float*>(smem + kSlabLds) + (inv == reinterpret_cast<float*>(smem + kSlabLds) ? 256 : 0);
            inv[row] = rsqrtf(ss / (float)a.K + a.eps);
        }
    };
    unsigned char* const stg = smem + kSlabRows + wave * 4096;
    const int c = lane % NCH, rr = lane / NCH;   // store phase: the lane's piece, its row within the RPS of an instruction
    auto epi = [&](auto NMC, int tile, int m, auto& acc) {
        constexpr int NM = decltype(NMC)::value;
        int tm, tn, sl;
        where(tile, tm, tn, sl);
        const int m0 = tm * TR + m + 16 * NM * wm;                      // the wave's first row
        const int ld = PAIR ? a.F : a.N, n = (PAIR ? tn * 128 : tn * 256) + OC * wn + 8 * c;
        u16x8 rv[MODE == kPPResid ? NK : 1];
        auto resid = [&](int t) {
            if constexpr (MODE == kPPResid) {
#pragma unroll
                for (int k = 0; k < NK; ++k)
                    rv[k] = *reinterpret_cast<const u16x8*>(a.resid + (int64_t)min(m0 + 16 * t + RPS * k + rr, a.M - 1) * ld + n);
            }
        };
        resid(0);
#pragma unroll
        for (int t = 0; t < NM; ++t) {
            // 16 rows at a time; accumulator (s, t): row 16 t + lane % 16, columns 16 s + 4 (lane / 16) .. + 3.  Row r's piece p lies at
            // p ^ (r % NCH)
            const int r = lane & 15;
            float sc = 1.f;
            if constexpr (NORMP) sc = inv[16 * NM * wm + 16 * t + r];
            if constexpr (MODE == kPPPart) {   // (two blocks of columns make a line)
                const int row = m0 + 16 * t + r;
#pragma unroll
                for (int s = 0; s < 8; ++s) {
                    const int col = tn * 256 + OC * wn + 16 * s + 4 * (lane >> 4);
                    if (row < a.M && col < a.N) *reinterpret_cast<f32x4*>(a.ws + ((int64_t)sl * a.M + row) * a.N + col) = acc[s][t] * sc;
                    acc[s][t] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
                continue;
            }
#pragma unroll
            for (int s = 0; s < (PAIR ? 4 : 8); ++s) {
                const int col = 16 * s + 4 * (lane >> 4);
                u16x4 o;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float v = acc[s][t][i] * sc;
                    if constexpr (MODE == kPPSwiglu) {
                        const float gv = bf2f(f2bf(v));
                        const float sg = bf2f(f2bf(gv / (1.f + __expf(-gv))));
                        o[i] = f2bf(sg * bf2f(f2bf(acc[s + 4][t][i] * sc)));
                    } else if constexpr (MODE == kPPGlu) {
                        const float gv = fminf(v, a.limit), u = fminf(fmaxf(acc[s + 4][t][i] * sc, -a.limit), a.limit);
                        o[i] = f2bf(gv * hy::sigmoid_act<uint16_t>(a.slope * gv) * (u + a.shift));
                    } else if constexpr (MODE == kPPRelu2 || MODE == kPPGelu) {
                        o[i] = f2bf(hy::act_apply(v, MODE == kPPRelu2 ? hy::kActRelu2 : hy::kActGelu));
                    } else {
                        o[i] = f2bf(v);
                    }
                }
                *reinterpret_cast<u16x4*>(stg + r * RBY + (((col >> 3) ^ (r % NCH)) << 4) + ((col >> 2) & 1) * 8) = o;
            }
#pragma unroll
            for (int s = 0; s < 8; ++s) acc[s][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            u16x8 v[NK];
#pragma unroll
            for (int k = 0; k < NK; ++k) {   // (a wave's LDS operations complete in order)
                const int q = RPS * k + rr;
                v[k] = *reinterpret_cast<const u16x8*>(stg + q * RBY + ((c ^ (q % NCH)) << 4));
            }
            float ss[NK];
            if constexpr (MODE == kPPResid) {
#pragma unroll
                for (int k = 0; k < NK; ++k) {
                    u16x8 o;
                    ss[k] = 0.f;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const float y = bf2f(f2bf(bf2f(v[k][i]) + bf2f(rv[k][i])));
                        o[i] = f2bf(y);
                        ss[k] += y * y;
                    }
                    v[k] = o;
                    ss[k] = row_sum16(ss[k]);
                }
                if (t + 1 < NM) resid(t + 1);
            }
#pragma unroll
            for (int k = 0; k < NK; ++k) {
                const int row = m0 + 16 * t + RPS * k + rr;
                if (row >= a.M) continue;
                uint16_t* y = a.y + (int64_t)row * ld + n;
                if (PAIR || MODE == kPPResid || n + 8 <= a.N) *reinterpret_cast<u16x8*>(y) = v[k];
                else if (n < a.N) *reinterpret_cast<u16x4*>(y) = u16x4{v[k][0], v[k][1], v[k][2], v[k][3]};   // (N % 4 == 0)
                if constexpr (MODE == kPPResid)
                    if (c == 0) a.part_out[(int64_t)row * (a.N / 128) + tn * 2 + wn] = ss[k];
            }
        }
    };
    slab_run<PAIR, NMX>(smem, mt * nt * S, tail, MODE == kPPPart ? a.kts : a.K / 64, a.x, (int)((int64_t)a.M * a.K * 2), (int)((int64_t)a.N * a.K * 2), off, scales, epi);
}

// y = the new residual stream: the S slices of 8 columns per thread in their order, the residual, RMSNorm partials per 128 columns
__global__ void __launch_bounds__(256) slab_sum_resid_kernel(const float* __restrict__ ws, const uint16_t* __restrict__ resid,
                                                             uint16_t* __restrict__ y, float* __restrict__ part, int64_t n, int S) {
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;   // (n % 256 == 0: 16 lanes leave or stay together)
    if (i >= n) return;
    const u16x8 rv = *reinterpret_cast<const u16x8*>(resid + i);
    f32x4 v0 = *reinterpret_cast<const f32x4*>(ws + i), v1 = *reinterpret_cast<const f32x4*>(ws + i + 4);
#pragma unroll 4
    for (int s = 1; s < S; ++s) {
        v0 += *reinterpret_cast<const f32x4*>(ws + s * n + i);
        v1 += *reinterpret_cast<const f32x4*>(ws + s * n + i + 4);
    }
    u16x8 o;
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float t = bf2f(f2bf(bf2f(f2bf(k < 4 ? v0[k & 3] : v1[k & 3])) + bf2f(rv[k])));
        o[k] = f2bf(t);
        ss += t * t;
    }
    *reinterpret_cast<u16x8*>(y + i) = o;
    ss = row_sum16(ss);
    if ((threadIdx.x & 15) == 0) part[i / 128] = ss;
}

// x rows of a tile, in 32s, for M rows and nt tiles of W rows (walked S times): 8, whose last round may be of halves, or 4 to 7 where the
// rounds of such tiles take less.  A round's time, in those of 256 x 256 tiles, is from 1 to 4 rounds of 28672 x 4096 (4 rows-in-32s: 69, 115, 167, 245
// us; 5: 74, 127, 186, 247; 6: 77, 140, 213; 7: 84, 155, 235; 8: 95, 185, 267, its halves behind a round 50).  us, 256-row tiles -> the rows picked:
// that shape at 272 rows 84.9 -> 72.7, 384 89.9 -> 79.1, 528 143 -> 124, 896 184 -> 169, 1152 244 -> 222; 4096 x 14336 in 4 slices at 528 81.8 ->
// 69.0, 640 85.6 -> 73.1, in 8 at 272 55.9 -> 46.8, in 2 at 1152 137 -> 116; 6144 x 4096 at 1600 79.0 -> 65.7.
// In one round all tiles alike are as good as halves or better, because the short last rows of slab_tail come behind all others, where no
// XCD has their W rows any more (4096 x 14336 in 4 slices at 384 rows 66.8, 63.3 as three tiles of 128 rows).
// (Beyond two rounds the chip's power decides, which rows that are not there cost too: 28672 x 4096 at 5130 rows 937, as 27 tiles of 192 946.)
int slab_rows(int M, int nt, int S) {
    constexpr float cost[] = {0.61f, 0.67f, 0.76f, 0.86f};
    const int tail = slab_tail(M, nt, S);
    int full, half;
    slab_split((tail > 0 ? M / 256 : (M + 255) / 256) * nt * S, tail, full, half);
    float best = (float)((full + kSlabCUs - 1) / kSlabCUs) + (full ? 0.57f : 0.63f) * ((half + kSlabCUs - 1) / kSlabCUs);
    int nm = 8;
    for (int n = 4; n < 8; ++n) {
        const int64_t tiles = (int64_t)((M + 32 * n - 1) / (32 * n)) * nt * S;
        const float t = cost[n - 4] * ((tiles + kSlabCUs - 1) / kSlabCUs);
        if (t < best * (best > 2.5f ? 0.94f : 0.97f)) best = t, nm = n;
    }
    return nm;
}

template <int MODE, bool NORMP, int NMX>
void slab_launch_rows(const PPArgs& a, int nt, int S, hipStream_t st) {
    constexpr int lds = kSlabLds + (NORMP ? 2048 : 0);
    const auto kern = gemm_slab_kernel<MODE, NORMP, NMX>;
    static const hipError_t once = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    (void)once;
    const int tail = NMX == 8 ? slab_tail(a.M, nt, S) : 0, tiles = (tail > 0 ? a.M / 256 : (a.M + 32 * NMX - 1) / (32 * NMX)) * nt * S;
    hipLaunchKernelGGL(kern, dim3(NMX == 8 ? slab_grid(tiles, tail) : tiles < kSlabCUs ? tiles : kSlabCUs), dim3(256), lds, st, a);
}

template <int MODE, bool NORMP>
void slab_launch(const PPArgs& a, hipStream_t st) {
    const bool pair = MODE == kPPSwiglu || MODE == kPPGlu;
    const int nt = pair ? a.F / 128 : (a.N + 255) / 256, S = MODE == kPPPart ? a.splitk : 1;
    switch (slab_rows(a.M, nt, S)) {
        case 4: slab_launch_rows<MODE, NORMP, 4>(a, nt, S, st); break;
        case 5: slab_launch_rows<MODE, NORMP, 5>(a, nt, S, st); break;
        case 6: slab_launch_rows<MODE, NORMP, 6>(a, nt, S, st); break;
        case 7: slab_launch_rows<MODE, NORMP, 7>(a, nt, S, st); break;
        default: slab_launch_rows<MODE, NORMP, 8>(a, nt, S, st);
    }
}

}  // namespace

bool launch_gemm_slab(int mode, bool normp, const PPArgs& a, hipStream_t st) {
    if (normp && mode != kPPPlain && mode != kPPSwiglu) return false;
    if (a.splitk > 1) {
        if (mode != kPPPlain && mode != kPPResid) return false;
        normp ? slab_launch<kPPPart, true>(a, st) : slab_launch<kPPPart, false>(a, st);
        const int64_t n = (int64_t)a.M * a.N;
        if (mode == kPPPlain) {
            if (a.y != nullptr) launch_gemm_slices(a.ws, a.y, n, a.splitk, st);   // (else the slices are what is wanted)
        } else slab_sum_resid_kernel<<<(unsigned)((n / 8 + 255) / 256), 256, 0, st>>>(a.ws, a.resid, a.y, a.part_out, n, a.splitk);
        return true;
    }
    switch (mode) {
        case kPPPlain: normp ? slab_launch<kPPPlain, true>(a, st) : slab_launch<kPPPlain, false>(a, st); return true;
        case kPPSwiglu: normp ? slab_launch<kPPSwiglu, true>(a, st) : slab_launch<kPPSwiglu, false>(a, st); return true;
        case kPPResid: slab_launch<kPPResid, false>(a, st); return true;
        case kPPGlu: slab_launch<kPPGlu, false>(a, st); return true;
        case kPPRelu2: slab_launch<kPPRelu2, false>(a, st); return true;
        case kPPGelu: slab_launch<kPPGelu, false>(a, st); return true;
        default: return false;
    }
}

}  // namespace chronos
