/* The form in which the kernels work out expf (device_math.h: the cubic by Horner's rule and scaled in its last
 * multiply-add, arguments beyond a float's range moved to a bound) against the oracle's, all 2^32 arguments. */
#include <math.h>
#include <pthread.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

float or_expf(float);

static inline float asfloat(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
static inline uint32_t asuint(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
static inline double asdouble(uint64_t u) { double d; memcpy(&d, &u, 8); return d; }
static inline uint64_t asuint64(double d) { uint64_t u; memcpy(&u, &d, 8); return u; }

static uint64_t tab[32]; /* bits(2^(i/32)) - (i << 47) */

static inline float kernel_exp(float x)
{
    const double inv_ln2_n = 0x1.71547652b82fep+0 * 32.0, shift = 0x1.8p+52;
    const double c0 = 0x1.c6af84b912394p-5 / 32 / 32 / 32, c1 = 0x1.ebfce50fac4f3p-3 / 32 / 32, c2 = 0x1.62e42ff0c52d6p-1 / 32;
    const double xd = (double)(x < -104.0f ? -104.0f : (x > 89.0f ? 89.0f : x));
    double kd = fma(inv_ln2_n, xd, shift);
    const uint32_t ki = (uint32_t)asuint64(kd);
    kd -= shift;
    const double r = fma(inv_ln2_n, xd, -kd);
    const double s = asdouble(tab[ki & 31u] + ((uint64_t)(ki << 15) << 32));
    return (float)fma(fma(r, fma(c0, r, c1), c2), r * s, s);
}

typedef struct { uint64_t lo, hi, differ; } job_t;

static void* run(void* p)
{
    job_t* j = p;
    for (uint64_t u = j->lo; u < j->hi; ++u) {
        const float x = asfloat((uint32_t)u);
        if (x == x)
            j->differ += asuint(kernel_exp(x)) != asuint(or_expf(x));
    }
    return 0;
}

int main(int argc, char** argv)
{
    enum { NT = 8 };
    pthread_t th[NT];
    job_t jobs[NT];
    /* the table as the kernels' source has it, one entry per argument */
    if (argc != 33)
        return 2;
    for (int i = 0; i < 32; ++i)
        if (sscanf(argv[1 + i], "%lx", (unsigned long*)&tab[i]) != 1)
            return 2;
    const uint64_t per = (1ull << 32) / NT;
    for (int i = 0; i < NT; ++i) {
        jobs[i] = (job_t){i * per, (i + 1) * per, 0};
        pthread_create(&th[i], 0, run, &jobs[i]);
    }
    uint64_t differ = 0;
    for (int i = 0; i < NT; ++i) {
        pthread_join(th[i], 0);
        differ += jobs[i].differ;
    }
    printf("differ %lu\n", (unsigned long)differ);
    return differ != 0;
}
