// The sum of a float row in the order of torch's CPU sum (SumKernel.cpp: under 8 elements four partial sums, else
// vectors of 8 in four partial sums, the tail first, the lanes of the vector last) for a row length that only the
// launch knows. Plain C++ (the host test compiles it with g++).
//
// Every element is read unconditionally, in blocks of 8, from a row that is padded with zeros to whole blocks, and the
// blocks that a length has are chosen by branches on the length alone. (One masked add per element, the form that
// this replaces, kept a lane mask per element and per call site alive over the whole step: 1066 spilled scalar
// registers in the Wi-Fi mean-field step at one AP, read back by lane reads in every sub-step, and 276 vector
// registers, one wavefront per SIMD; the present step spills 164 and has 175, two wavefronts. 2048 envs of 16 robots,
// one env per wavefront: 437 us a step before, 278 after.) A zero added to a partial sum changes no bit of the result:
// the last sum begins at +0.0, so none of it is -0.0.
#pragma once

#ifdef __HIPCC__
#define ROW_FN __device__ __forceinline__
#else
#define ROW_FN inline
#endif

namespace inet {

// eight consecutive elements (a vector type: arrays went to scratch memory where many sums are inlined)
typedef float Row8 __attribute__((vector_size(32)));

// n = 1 .. 71. x(i): element i; blk(b): elements 8 b .. 8 b + 7, zeros past the row's end. Only blocks that
// hold an element of the row are read; below 8 elements, x(0), x(1), with n > 2 also x(2), x(3), with n > 4 up to x(6).
template <class X, class B>
ROW_FN float aten_sum_padded(int n, X x, B blk) {
    if (n < 8) {
        float s = 0.0f + x(0);
        const float x1 = x(1);
        if (n > 4) {
            const float x4 = x(4), x5 = x(5), x6 = x(6);
            s += x4;
            s += x5;
            s += x6;
        }
        s += x1;
        if (n > 2) {
            const float x2 = x(2), x3 = x(3);
            s += x2;
            s += x3;
        }
        return s;
    }
    const int nv = n >> 3, nt = n & 7;
    Row8 a = blk(0);
    float fin = 0.0f;
    if (nt > 0) {
        const Row8 v = blk(nv);
        fin += v[0];
        if (nt > 1) {
            fin += v[1];
            fin += v[2];
            if (nt > 3) {
                fin += v[3];
                fin += v[4];
                fin += v[5];
                fin += v[6];
            }
        }
    }
    if (nv < 4) {                       // (one partial sum per vector lane)
        if (nv > 1) a += blk(1);
        if (nv > 2) a += blk(2);
    } else {                            // (vectors 4 .. 7 into the first partial sum, or one into each with eight)
        if (nv > 4) a += blk(4);
        if (nv == 8) {
            a += blk(1) + blk(5);
            a += blk(2) + blk(6);
            a += blk(3) + blk(7);
        } else {
            if (nv > 5) a += blk(5);
            if (nv > 6) a += blk(6);
            a += blk(1);
            a += blk(2);
            a += blk(3);
        }
    }
    fin += a[0];
    fin += a[1];
    fin += a[2];
    fin += a[3];
    fin += a[4];
    fin += a[5];
    fin += a[6];
    fin += a[7];
    return fin;
}

}  // namespace inet
