// pivot_step.hpp -- the pivot search of one column over a workgroup.
//
// A column step of the register-resident panels is a chain of dependent
// cross-lane operations, so their number is what it costs:
//   * within a wavefront the largest key word (the high word of an FP64 key)
//     is found by six DPP maxima; when exactly one lane holds it -- the usual
//     case -- that lane is the candidate and the full (key, row) reduction is
//     skipped;
//   * the candidate's value, key word and row go to LDS as one 16-byte
//     record; after a barrier lane w of every wavefront reads record w, forms
//     its reciprocal while the maximum over the records is taken, and the
//     winner's fields are read from its lane.
// The pivot row itself goes to LDS after the choice, by the one thread that
// holds it, before a second barrier.  Against every wavefront publishing its
// candidate row before a single barrier: FP64 LU n = 256 x 4096 4.18 -> 3.79
// ms, n = 300 x 1024 2.96 -> 2.43, n = 128 x 16384 3.06 -> 2.86; FP32 n = 256
// x 4096 1.81 -> 1.63 ms.  A batch of 64 FP32 matrices of n = 96, latency
// alone, lost 3 us to the second barrier and takes 71 us since the diagonal
// blocks are inverted by four lanes per column (78 before both).  Putting off the update of the columns beyond the next
// one until after the search's barrier was slower (n = 2000 5.08 -> 5.24 ms).
#pragma once

#include "common.hpp"

namespace rsa
{

struct alignas(16) PivotRecord
{
    unsigned lo, hi; // the value's bits (FP32: lo)
    int word; // high word of its key (FP32: the key), -1: no candidate
    int row; // logical row
};

// largest signed integer over the wavefront, uniform
__device__ __forceinline__ int wave_max_uniform(int v)
{
    auto mx = [](int a, int b) { return a > b ? a : b; };
    v = mx(v, dpp_mov<0xB1>(v));
    v = mx(v, dpp_mov<0x4E>(v));
    v = mx(v, dpp_mov<0x141>(v));
    v = mx(v, dpp_mov<0x140>(v));
    // row_bcast:15 into rows 1 and 3, row_bcast:31 into rows 2 and 3
    v = mx(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xA, 0xF, false));
    v = mx(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xC, 0xF, false));
    return __builtin_amdgcn_readlane(v, 63);
}

// largest over groups of NW (1, 2, 4 or 8) consecutive lanes, in every lane
template <int NW>
__device__ __forceinline__ int few_max(int v)
{
    auto mx = [](int a, int b) { return a > b ? a : b; };
    if(NW > 1)
        v = mx(v, dpp_mov<0xB1>(v));
    if(NW > 2)
        v = mx(v, dpp_mov<0x4E>(v));
    if(NW > 4)
        v = mx(v, dpp_mov<0x141>(v));
    return v;
}
template <int NW>
__device__ __forceinline__ int few_min(int v)
{
    auto mn = [](int a, int b) { return a < b ? a : b; };
    if(NW > 1)
        v = mn(v, dpp_mov<0xB1>(v));
    if(NW > 2)
        v = mn(v, dpp_mov<0x4E>(v));
    if(NW > 4)
        v = mn(v, dpp_mov<0x141>(v));
    return v;
}

__device__ __forceinline__ int key_word(double k)
{
    return __double2hiint(k);
}
__device__ __forceinline__ int key_word(float k)
{
    return __float_as_int(k);
}

// This wavefront's candidate for the pivot of a column to *rec: key, val and
// row are the lane's own best (key: pivot_key, negative for none).
template <typename T>
__device__ __forceinline__ void publish_candidate(T key, T val, int row, PivotRecord* rec)
{
    const bool cand = key >= T(0);
    const int word = cand ? key_word(key) : -1;
    const int top = wave_max_uniform(word);
    bool mine = word == top;
    const uint64_t hit = __builtin_amdgcn_ballot_w64(mine);
    if((hit & (hit - 1)) != 0) // uniform: more than one lane holds the largest word
    {
        T k2 = key;
        int r2 = cand ? row : 0x7fffffff;
        wave_argmax(k2, r2);
        mine = cand ? row == r2 : r2 == 0x7fffffff; // no candidate: any lane's record
    }
    if(mine)
    {
        PivotRecord r;
        if constexpr(sizeof(T) == 8)
        {
            r.lo = unsigned(__double2loint(val));
            r.hi = unsigned(__double2hiint(val));
        }
        else
        {
            r.lo = __float_as_uint(val);
            r.hi = 0;
        }
        r.word = word;
        r.row = row;
        *rec = r;
    }
}

// The winner among the NW records of a column (at least one holds a
// candidate): largest key, ties to the lower row.  row and wave are uniform;
// the winner's value and its reciprocal are v and q of lane `wave`, read by
// the caller when it needs them (the division is then in flight under the
// pivot row's way through LDS).
template <typename T, int NW>
__device__ __forceinline__ void select_candidate(const PivotRecord* recs, int& row, int& wave,
                                                 T& v, T& q)
{
    const int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    const PivotRecord r = recs[lane & (NW - 1)];
    if constexpr(sizeof(T) == 8)
        v = __hiloint2double(int(r.hi), int(r.lo));
    else
        v = __uint_as_float(r.lo);
    q = T(1) / v;
    const int top = few_max<NW>(r.word);
    constexpr uint64_t MASK = NW == 64 ? ~0ull : (1ull << NW) - 1;
    uint64_t hit = __builtin_amdgcn_ballot_w64(r.word == top) & MASK;
    if((hit & (hit - 1)) != 0) // uniform
    {
        bool tied = r.word == top;
        if constexpr(sizeof(T) == 8)
        {
            // low words, shifted to order as signed integers; a NaN's key is +inf
            const int low = isnan_t(v) ? int(0x80000000u) : int(r.lo ^ 0x80000000u);
            const int most = few_max<NW>(tied ? low : int(0x80000000u));
            tied = tied && low == most;
        }
        const int first = few_min<NW>(tied ? r.row : 0x7fffffff);
        hit = __builtin_amdgcn_ballot_w64(tied && r.row == first) & MASK;
    }
    wave = __builtin_ctzll(hit);
    row = __builtin_amdgcn_readlane(r.row, wave);
}

} // namespace rsa
