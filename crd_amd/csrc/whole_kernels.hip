// The long one-kernel transforms of gfx950: n = 2^15 and 2^16 C2C in one launch, each transform held by one
// workgroup from its load to its store.
//
// A CU's register file is 512 KiB and its LDS 160 KiB, so one 512-thread workgroup (256 registers per lane) can keep a
// whole 2^16-point transform (512 KiB): three quarters in registers, a quarter in LDS. The four-step's intermediate
// then never leaves the CU and every point crosses the L2 boundary twice (16 bytes) instead of four times.
//
// n = 256 x N2 (N2 = 32 NT, NT = 4 or 8 column tiles of 32).
//   columns  per tile: thread (lc = tid % 32, li = tid / 32) loads x[(li + 16 m) N2 + 32 tile + lc], m < 16 (runs of
//            256 bytes); a radix-16 pass over m, an exchange through 32 KiB of LDS (real parts, then imaginary parts)
//            that also turns the threads to (i = tid % 16, c = tid / 16), the second radix-16 pass, the four-step
//            twiddle W_n^{col k1} (its table transposed: 128-byte runs). The thread then holds column 32 tile + c at
//            k1 = i + 16 m, again as 16 values, in the registers the tile was loaded into (or, for LT tiles, in LDS
//            slots of its own that no other thread reads).
//   rows     per set of 16 rows (one m, or two of them when NT = 4): 8 values per thread are a register DFT over the
//            tiles; of the 32 points left over c = 4 a + b, a is the wave and b the lane's upper bits: a radix-8 pass
//            over a after an exchange of registers against waves through LDS, a radix-4 pass over b after a swap of
//            registers against lane bits. The 16 rows sit on adjacent lanes, so every store is a run of 128 bytes.
// The registers of a row set are free once it is read, so the next transform's loads go into them at once: they
// are in flight during the rest of the row phase. The grid is at most one workgroup per CU; workgroup b runs transforms
// b, b + grid, ...
//
// Measured (MI355X): n = 2^16 x 2048 0.691 (two four-step passes) -> 0.490 ms, 4.4 TB/s; x 4096 1.39 -> 0.93 ms;
// n = 2^15 x 4096 0.712 -> 0.445 ms, 4.8 TB/s; rel-L2 against FP64 1.45e-7 and 1.39e-7 as before. A round of 256
// transforms of 2^16 takes 58 us against 43 us for its bytes at the copy rate: what is left is the column phase, whose
// LDS exchanges and L2 twiddle reads two waves per SIMD hide only in part (VALU about 40 % busy).
// What shaped it, at 2^16 x 2048 / 2^15 x 4096: rows kept in lane order through two LDS exchanges per row set 0.615 ms
// / -; the 16 rows on adjacent lanes and one of the exchanges as lane swaps 0.586 / 0.536; each exchange beside the
// arithmetic of the tile or set before and after it, wide exchange spaces 0.548 / 0.498; starts spread within an XCD
// (see launch) 0.490 / 0.445.
#include "buffer.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace crdfft
{
using namespace dev;

namespace
{

template <int NT> struct WholeCfg
{
    static_assert(NT == 4 || NT == 8, "n = 2^15 or 2^16");
    static constexpr int N1 = 256, N2 = 32 * NT;
    static constexpr uint32_t N = N1 * N2;
    static constexpr int threads = 512;
    static constexpr int LT = NT == 8 ? 2 : 0; // column tiles kept in LDS between the two phases
    static constexpr int ST = NT - LT;         // column tiles kept in registers
    // exchange space from 0. Wide: whole points, 16 rows of 512 at a pitch of 513; NT = 4 alternates between two of
    // them (one barrier each). Narrow: 16 rows of 512 floats at a pitch of 514, real parts then imaginary parts. The
    // pitches put the lanes of one access on different banks. The row exchange takes 8 x 512 points.
    static constexpr int wide_pitch = 513, wide_bytes = 16 * wide_pitch * 8;
    static constexpr int narrow_pitch = 514, narrow_bytes = 16 * narrow_pitch * 4;
    static constexpr bool two_wide = LT == 0;
    // stage twiddles W_256^{i m}, m = 1..15, and W_256^{c q}, q = 1..7
    static constexpr int t1_points = 15 * 16, t2_points = 7 * 32;
    // kept tiles: values of tile S + 1 (all but the last one, which stays in a register) behind the narrow space, over
    // the wide one; those of tile S behind it
    static constexpr int keep1_off = narrow_bytes;
    static constexpr int keep0_off = keep1_off + 15 * threads * 8;
    static constexpr int tab_off = two_wide ? 2 * wide_bytes : keep0_off + 16 * threads * 8;
    static constexpr int lds_bytes = tab_off + (t1_points + t2_points) * 8;
    static_assert(narrow_bytes >= 8 * threads * 8, "the row exchange fits the narrow space");
    static_assert(two_wide || keep0_off >= wide_bytes, "the first kept tile is clear of the wide space");
    static_assert(lds_bytes <= 160 * 1024, "LDS of a CU");
};

__device__ __forceinline__ void lane_swap32(float& x, float& y)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, y),
                                                    false, false);
    x = __builtin_bit_cast(float, static_cast<uint32_t>(r[0]));
    y = __builtin_bit_cast(float, static_cast<uint32_t>(r[1]));
}

__device__ __forceinline__ void lane_swap16(float& x, float& y)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, y),
                                                    false, false);
    x = __builtin_bit_cast(float, static_cast<uint32_t>(r[0]));
    y = __builtin_bit_cast(float, static_cast<uint32_t>(r[1]));
}

// A radix-16 DFT in two halves (the same arithmetic as Dft<16>): four radix-4 DFTs and the inner twiddles, then four
// more. In between, value k1 of the DFT over a[4 n1 + n2] sits at a[4 k1 + n2].
template <bool INV> struct Dft16Halves
{
    template <int N2, int... K1> static __device__ __forceinline__ void twiddle(cf* t, std::integer_sequence<int, K1...>)
    {
        ((t[K1] = twc<static_cast<long>(N2) * K1, 16, INV>(t[K1])), ...);
    }
    template <int N2> static __device__ __forceinline__ void column(cf* a)
    {
        cf t[4] = {a[N2], a[4 + N2], a[8 + N2], a[12 + N2]};
        Dft<4, INV>::run(t);
        twiddle<N2>(t, std::make_integer_sequence<int, 4>{});
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            a[4 * k + N2] = t[k];
        }
    }
    static __device__ __forceinline__ void first(cf* a)
    {
        column<0>(a);
        column<1>(a);
        column<2>(a);
        column<3>(a);
    }
    static __device__ __forceinline__ void second(cf* a)
    {
        cf t[16];
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1)
        {
            cf u[4] = {a[4 * k1], a[4 * k1 + 1], a[4 * k1 + 2], a[4 * k1 + 3]};
            Dft<4, INV>::run(u);
#pragma unroll
            for (int k2 = 0; k2 < 4; ++k2)
            {
                t[k1 + 4 * k2] = u[k2];
            }
        }
#pragma unroll
        for (int k = 0; k < 16; ++k)
        {
            a[k] = t[k];
        }
    }
};

// The segments between two barriers keep their instructions (the scheduler would gather the arithmetic after the last
// barrier and leave the LDS waits bare).
__device__ __forceinline__ void segment_barrier()
{
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
}

// The second half of a column tile: v holds the exchanged values (index m of thread i) and leaves with the twiddled X
// at k1 = i + 16 m of column 32 tile + c.
template <int NT, bool INV>
__device__ __forceinline__ void column_finish(cf (&v)[16], int tile, const cf* t1, __amdgpu_buffer_rsrc_t tfull)
{
    const int tid = threadIdx.x;
    const int i = tid & 15;
    const uint32_t voff = static_cast<uint32_t>(i + 256 * (tid >> 4)) * 8u;
#pragma unroll
    for (int m = 1; m < 16; ++m)
    {
        v[m] = ctw<INV>(v[m], t1[(m - 1) * 16 + i]);
    }
    Dft<16, INV>::run(v);
#pragma unroll
    for (int m = 0; m < 16; ++m)
    {
        v[m] = ctw<INV>(v[m], bld<0>(tfull, voff, static_cast<uint32_t>(16 * m + 256 * 32 * tile) * 8u));
    }
}

// Column phase, tile `v` (after its first radix-16 pass) through the exchange space at `lds` while `fin` finishes the
// tile before it and the next tile's first pass runs in `nx`. TAIL: the space is free for anyone on return.
template <int NT, bool INV, bool WIDE, bool TAIL, bool NEXT, class Fin>
__device__ __forceinline__ void column_exchange(cf (&v)[16], cf (&nx)[16], char* lds, Fin fin)
{
    using C = WholeCfg<NT>;
    const int tid = threadIdx.x;
    if constexpr (WIDE)
    {
        cf* const ex = reinterpret_cast<cf*>(lds);
        cf* const wr = ex + tid;                                            // (k, li, lc) at k pitch + 32 li + lc
        const cf* const rd = ex + (tid & 15) * C::wide_pitch + (tid >> 4);  // (i, m, c)
#pragma unroll
        for (int k = 0; k < 16; ++k)
        {
            wr[k * C::wide_pitch] = v[k];
        }
        fin();
        segment_barrier();
#pragma unroll
        for (int m = 0; m < 16; ++m)
        {
            v[m] = rd[m * 32];
        }
        if constexpr (NEXT)
        {
            Dft16Halves<INV>::first(nx);
            Dft16Halves<INV>::second(nx);
        }
    }
    else
    {
        float* const ex = reinterpret_cast<float*>(lds);
        float* const wr = ex + tid;
        const float* const rd = ex + (tid & 15) * C::narrow_pitch + (tid >> 4);
#pragma unroll
        for (int k = 0; k < 16; ++k)
        {
            wr[k * C::narrow_pitch] = v[k].x;
        }
        fin();
        segment_barrier();
#pragma unroll
        for (int m = 0; m < 16; ++m)
        {
            v[m].x = rd[m * 32];
        }
        if constexpr (NEXT)
        {
            Dft16Halves<INV>::first(nx);
        }
        segment_barrier();
#pragma unroll
        for (int k = 0; k < 16; ++k)
        {
            wr[k * C::narrow_pitch] = v[k].y;
        }
        segment_barrier();
#pragma unroll
        for (int m = 0; m < 16; ++m)
        {
            v[m].y = rd[m * 32];
        }
        if constexpr (NEXT)
        {
            Dft16Halves<INV>::second(nx);
        }
    }
    if constexpr (TAIL)
    {
        segment_barrier();
    }
    else
    {
        __builtin_amdgcn_sched_barrier(0);
    }
}

template <int NT, bool INV> __global__ __launch_bounds__(512) void k_whole(WholeArgs a)
{
    using C = WholeCfg<NT>;
    constexpr int S = C::ST;
    constexpr int RM = 8 / NT; // values of m per row set
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    cf* const keep0 = reinterpret_cast<cf*>(lds_raw + C::keep0_off) + threadIdx.x; // value m at [512 m]
    cf* const keep1 = reinterpret_cast<cf*>(lds_raw + C::keep1_off) + threadIdx.x;
    cf* const t1 = reinterpret_cast<cf*>(lds_raw + C::tab_off); // W_256^{i m} at [(m - 1) 16 + i]
    cf* const t2 = t1 + C::t1_points;                           // W_256^{c q} at [(q - 1) 32 + c]
    const int tid = threadIdx.x;
    const int i = tid & 15;
    const int c = tid >> 4;
    const int b = c & 3;
    const int w = tid >> 6; // wave
    {
        const cf* roots = reinterpret_cast<const cf*>(a.roots); // W_256^e
        if (tid < C::t1_points)
        {
            t1[tid] = roots[((tid >> 4) + 1) * (tid & 15)]; // at most 15 * 15
        }
        if (tid < C::t2_points)
        {
            t2[tid] = roots[((tid >> 5) + 1) * (tid & 31)]; // at most 7 * 31
        }
    }
    __syncthreads();
    const __amdgpu_buffer_rsrc_t tfull = make_rsrc(a.tfull, C::N * 8u);
    const uint32_t load_off = static_cast<uint32_t>((tid >> 5) * C::N2 + (tid & 31)) * 8u;
    // output i + 16 m + 256 (q + NT s + 8 NT u): wave w holds q = w % NT (of row m0 + w / NT), the lane s = 4 h + b
    const uint32_t store_off = static_cast<uint32_t>(i + 16 * (w / NT) + 256 * (w % NT + NT * b)) * 8u;

    for (uint32_t d = ((blockIdx.x >> 3) & 31u) * a.stagger; d > 0; --d)
    {
        __builtin_amdgcn_s_sleep(16); // 1024 clocks
    }
    uint64_t t = blockIdx.x;
    cf s[S][16];
    cf last{};
    // slots S - LT + l first hold the LDS tiles (numbers S + l), then their own
    {
        const __amdgpu_buffer_rsrc_t src = make_rsrc(reinterpret_cast<const cf*>(a.in) + t * a.idist, C::N * 8u);
#pragma unroll
        for (int m = 0; m < 16; ++m)
        {
#pragma unroll
            for (int q = 0; q < S; ++q)
            {
                const int tile = q < S - C::LT ? q : q + C::LT;
                s[q][m] = bld<kAuxNt>(src, load_off, static_cast<uint32_t>(16 * m * C::N2 + 32 * tile) * 8u);
            }
        }
    }
#pragma unroll 1
    for (; t < a.count; t += gridDim.x)
    {
        const __amdgpu_buffer_rsrc_t src = make_rsrc(reinterpret_cast<const cf*>(a.in) + t * a.idist, C::N * 8u);
        if constexpr (C::LT > 0)
        {
            // column phase: tile 6 (kept in LDS) from slot 4, tiles 0-2, tile 7 (kept) from slot 5, tile 3, then tiles
            // 4 and 5, loaded into slots 4 and 5 as soon as those are free. The wide space is there until tile 7 is
            // kept.
            static_assert(NT == 8 && S == 6, "the order below");
            auto reload = [&](int q) {
#pragma unroll
                for (int m = 0; m < 16; ++m)
                {
                    s[q][m] = bld<kAuxNt>(src, load_off, static_cast<uint32_t>(16 * m * C::N2 + 32 * q) * 8u);
                }
            };
            Dft<16, INV>::run(s[4]);
            column_exchange<NT, INV, true, true, true>(s[4], s[0], lds_raw, [] {});
            column_exchange<NT, INV, true, true, true>(s[0], s[1], lds_raw, [&] {
                column_finish<NT, INV>(s[4], 6, t1, tfull);
#pragma unroll
                for (int m = 0; m < 16; ++m)
                {
                    keep0[m * C::threads] = s[4][m];
                }
                reload(4);
            });
            column_exchange<NT, INV, true, true, true>(s[1], s[2], lds_raw,
                                                       [&] { column_finish<NT, INV>(s[0], 0, t1, tfull); });
            column_exchange<NT, INV, true, true, true>(s[2], s[5], lds_raw,
                                                       [&] { column_finish<NT, INV>(s[1], 1, t1, tfull); });
            column_exchange<NT, INV, true, true, true>(s[5], s[3], lds_raw,
                                                       [&] { column_finish<NT, INV>(s[2], 2, t1, tfull); });
            column_exchange<NT, INV, false, true, true>(s[3], s[4], lds_raw, [&] {
                column_finish<NT, INV>(s[5], 7, t1, tfull);
#pragma unroll
                for (int m = 0; m < 15; ++m)
                {
                    keep1[m * C::threads] = s[5][m];
                }
                last = s[5][15];
                reload(5);
            });
            column_exchange<NT, INV, false, true, true>(s[4], s[5], lds_raw,
                                                        [&] { column_finish<NT, INV>(s[3], 3, t1, tfull); });
            column_exchange<NT, INV, false, true, false>(s[5], s[5], lds_raw,
                                                         [&] { column_finish<NT, INV>(s[4], 4, t1, tfull); });
            column_finish<NT, INV>(s[5], 5, t1, tfull);
        }
        else
        {
            // column phase: tiles 0 .. S - 1, alternating between the two wide spaces
            Dft<16, INV>::run(s[0]);
            column_exchange<NT, INV, true, false, true>(s[0], s[1], lds_raw, [] {});
#pragma unroll
            for (int q = 1; q < S; ++q)
            {
                char* const space = lds_raw + (q & 1) * C::wide_bytes;
                auto fin = [&] { column_finish<NT, INV>(s[q - 1], q - 1, t1, tfull); };
                if (q + 1 < S)
                {
                    column_exchange<NT, INV, true, false, true>(s[q], s[q + 1 < S ? q + 1 : q], space, fin);
                }
                else
                {
                    column_exchange<NT, INV, true, false, false>(s[q], s[q], space, fin);
                }
            }
            column_finish<NT, INV>(s[S - 1], S - 1, t1, tfull);
        }
        // the next transform of this workgroup (no records when there is none: its loads return zeros)
        const bool more = t + gridDim.x < a.count;
        const __amdgpu_buffer_rsrc_t nsrc =
            make_rsrc(reinterpret_cast<const cf*>(a.in) + (more ? t + gridDim.x : t) * a.idist, more ? C::N * 8u : 0u);
        const __amdgpu_buffer_rsrc_t dst = make_rsrc(reinterpret_cast<cf*>(a.out) + t * a.odist, C::N * 8u);
        cf u[8], y[8];
        // row set m0: values of its rows, first pass and twiddle, into u[m' NT + q]
        auto rows_first = [&](int m0) {
#pragma unroll
            for (int mm = 0; mm < RM; ++mm)
            {
#pragma unroll
                for (int q = 0; q < S; ++q)
                {
                    u[mm * NT + q] = s[q][m0 + mm];
                }
                if constexpr (C::LT > 0)
                {
                    u[S] = keep0[m0 * C::threads];
                    u[S + 1] = m0 < 15 ? keep1[m0 * C::threads] : last;
                }
                Dft<NT, INV>::run(u + mm * NT);
#pragma unroll
                for (int q = 1; q < NT; ++q)
                {
                    u[mm * NT + q] = ctw<INV>(u[mm * NT + q], t2[(q * (8 / NT) - 1) * 32 + c]); // W_N2^{c q}
                }
            }
        };
        // the next transform's points for the registers of row set m0
        auto prefetch = [&](int m0) {
#pragma unroll
            for (int mm = 0; mm < RM; ++mm)
            {
#pragma unroll
                for (int q = 0; q < S; ++q)
                {
                    const int tile = q < S - C::LT ? q : q + C::LT;
                    s[q][m0 + mm] =
                        bld<kAuxNt>(nsrc, load_off, static_cast<uint32_t>(16 * (m0 + mm) * C::N2 + 32 * tile) * 8u);
                }
            }
        };
        // row set m0 after its exchange (in y): the last two passes and the store
        auto rows_last = [&](int m0) {
            Dft<8, INV>::run(y);
#pragma unroll
            for (int e = 1; e < 8; ++e)
            {
                y[e] = ctw<INV>(y[e], t2[(e - 1) * 32 + 8 * b]); // W_32^{b e}
            }
            // the low two bits of s (registers) <-> b (lane bits 4 and 5)
#pragma unroll
            for (int e = 0; e < 8; ++e)
            {
                if ((e & 2) == 0)
                {
                    lane_swap32(y[e].x, y[e + 2].x);
                    lane_swap32(y[e].y, y[e + 2].y);
                }
            }
#pragma unroll
            for (int e = 0; e < 8; e += 2)
            {
                lane_swap16(y[e].x, y[e + 1].x);
                lane_swap16(y[e].y, y[e + 1].y);
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
            {
                Dft<4, INV>::run(y + h * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                {
                    const cf o = {y[h * 4 + e].x * a.scale, y[h * 4 + e].y * a.scale};
                    bst<kAuxNt>(dst, store_off, static_cast<uint32_t>(16 * m0 + 256 * (4 * NT * h + 8 * NT * e)) * 8u, o);
                }
            }
        };
        rows_first(0);
#pragma unroll
        for (int m0 = 0; m0 < 16; m0 += RM)
        {
            // register r of wave w <-> register w of wave r; the set before finishes beside the writes, the set after
            // starts beside the reads
            cf* const exc = reinterpret_cast<cf*>(lds_raw + (C::two_wide ? (m0 / RM & 1) * C::wide_bytes : 0));
#pragma unroll
            for (int r = 0; r < 8; ++r)
            {
                exc[r * 512 + tid] = u[r];
            }
            prefetch(m0);
            if (m0 > 0)
            {
                rows_last(m0 - RM);
            }
            segment_barrier();
#pragma unroll
            for (int e = 0; e < 8; ++e)
            {
                y[e] = exc[w * 512 + e * 64 + (tid & 63)];
            }
            if (m0 + RM < 16)
            {
                rows_first(m0 + RM);
            }
            if constexpr (C::two_wide)
            {
                __builtin_amdgcn_sched_barrier(0);
            }
            else
            {
                segment_barrier();
            }
        }
        rows_last(16 - RM);
    }
}

// The start of the workgroups of an XCD is spread over 31 * stagger * 1024 clocks: in step, all CUs load and store in
// the row phase at once and leave the memory idle in the column phase.
template <int NT, bool INV> hipError_t launch(WholeArgs a, unsigned grid, hipStream_t s)
{
    const uint64_t rounds = a.count / grid;
    a.stagger = NT == 8 ? (rounds >= 4 ? 2u : 1u) : (rounds >= 4 ? 1u : 0u);

    using C = WholeCfg<NT>;
    auto kern = k_whole<NT, INV>;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, C::lds_bytes);
    if (e != hipSuccess)
    {
        return e;
    }
    hipLaunchKernelGGL(kern, dim3(grid), dim3(C::threads), C::lds_bytes, s, a);
    return hipGetLastError();
}

} // namespace

bool whole_kernel_n(uint64_t n, uint64_t* n2)
{
    if (n != WholeCfg<4>::N && n != WholeCfg<8>::N)
    {
        return false;
    }
    *n2 = n / 256;
    return true;
}

hipError_t launch_whole(uint64_t n, bool inverse, const WholeArgs& a, unsigned grid, hipStream_t s)
{
    if (a.count == 0)
    {
        return hipSuccess;
    }
    grid = static_cast<unsigned>(std::min<uint64_t>(grid, a.count));

    if (grid == 0 || a.tfull == nullptr || a.roots == nullptr)
    {
        return hipErrorInvalidValue;
    }
    if (n == WholeCfg<4>::N)
    {
        return inverse ? launch<4, true>(a, grid, s) : launch<4, false>(a, grid, s);
    }
    if (n == WholeCfg<8>::N)
    {
        return inverse ? launch<8, true>(a, grid, s) : launch<8, false>(a, grid, s);
    }
    return hipErrorInvalidValue;
}

} // namespace crdfft
