/* Upper bounds of the simplex noise n over all positions in a simplex and all
 * gradients at its corners, proven by branch and bound over positions: |n|,
 * |grad n| and the norm of the Hessian.
 *
 * For a unit vector u each of n, u . grad n and u^T H u is a sum over the four
 * corners of g . w, g the corner's gradient (one of the twelve (+-1, +-1, 0) and
 * permutations).  With d the offset from the corner, s = d . d, r = sqrt s,
 * t = max(1/2 - s, 0), q = d . u, times 76.8:
 *   n             w = t^4 d
 *   u . grad n    w = t^4 u - 8 t^3 q d
 *   u^T H u       w = -16 t^3 q u + (48 t^2 q^2 - 8 t^3) d
 * The largest g . w is the two largest |components| of w added, which changes
 * by at most sqrt 2 |dw|, and |dw| is at most |dx| times
 *   n             t^4 + 8 t^3 s
 *   u . grad n    24 t^3 r + 48 t^2 s r
 *   u^T H u       24 t^3 + 288 t^2 s + 192 t s^2
 * (|grad t| = 2 r, |q| <= r, |grad q| = 1).
 *
 * Directions: of a set that leaves none further than theta from one of its
 * own, the best falls short of the norm by the factor cos theta for a vector
 * (u . grad n) and by no more than cos^2 theta - sin^2 theta for a symmetric
 * matrix.  A cell is done when the largest of a coarse or a fine set at its
 * centre and the change within it, over that factor, stay below the limit;
 * otherwise it is halved.
 *
 *   noise_bounds WHICH LIMIT    prints the largest value seen and the cells;
 *                               0: proven, 1: a value above, 2: too many cells or too small ones
 */
#include <math.h>
#include <stdio.h>
#include <stdlib.h>

#define ROOT2 1.4142135623730951
#define ROOT3 1.7320508075688772
#define COARSE 10
#define FINE 24
static const double corner[4][3] = {{0, 0, 0}, {1, 0, 0}, {1, 1, 0}, {1, 1, 1}};
static const long most = 200000000;
static int which, state;
static double limit, best;
static long cells;

struct dirs {
    int n;
    double factor, u[3][3 * FINE * FINE];
};
static struct dirs sets[2];

/* the points of an n x n grid on three faces of a cube, normalised: in the plane no point is further than
 * sqrt 2 / n from one, and normalising brings points together */
static void fill(struct dirs *s, int n) {
    const double theta = ROOT2 / n;
    s->n = 0;
    for (int f = 0; f < 3; f++)
        for (int i = 0; i < n; i++)
            for (int j = 0; j < n; j++) {
                const double a = (2 * i + 1.0) / n - 1, b = (2 * j + 1.0) / n - 1, len = sqrt(1 + a * a + b * b);
                s->u[f][s->n] = 1 / len;
                s->u[(f + 1) % 3][s->n] = a / len;
                s->u[(f + 2) % 3][s->n++] = b / len;
            }
    s->factor = which == 2 ? 1 - 2 * theta * theta : which == 1 ? 1 - theta * theta / 2 : 1;
    if (!which) s->n = 1;
}

static double largest(const struct dirs *s, const double (*d)[3], const double *t) {
    double sum[3 * FINE * FINE], top = 0;
    for (int i = 0; i < s->n; i++) sum[i] = 0;
    for (int k = 0; k < 4; k++) {
        const double t2 = t[k] * t[k], t3 = t2 * t[k], t4 = t2 * t2, dx = d[k][0], dy = d[k][1], dz = d[k][2];
        if (t[k] == 0) continue;
        for (int i = 0; i < s->n; i++) {
            const double q = dx * s->u[0][i] + dy * s->u[1][i] + dz * s->u[2][i];
            const double on_u = which == 0 ? 0 : which == 1 ? t4 : -16 * t3 * q;
            const double on_d = which == 0 ? t4 : which == 1 ? -8 * t3 * q : 48 * t2 * q * q - 8 * t3;
            const double a = fabs(on_u * s->u[0][i] + on_d * dx), b = fabs(on_u * s->u[1][i] + on_d * dy),
                         c = fabs(on_u * s->u[2][i] + on_d * dz);
            const double ab = a < b ? a : b;
            sum[i] += a + b + c - (ab < c ? ab : c);
        }
    }
    for (int i = 0; i < s->n; i++) top = sum[i] > top ? sum[i] : top;
    return 76.8 * top;
}

static void visit(const double x[3], double hx, long *count, double *seen) {
    if (state) return;
    if (++*count > most / 64 || hx < 1e-9) {
        state = 2;
        return;
    }
    const double rx = ROOT3 * hx;
    /* the simplex is 1 >= X >= Y >= Z >= 0 in skewed coordinates; none of the
     * differences changes by more than 2 |dx| */
    const double sk = (x[0] + x[1] + x[2]) / 3, X = x[0] + sk, Y = x[1] + sk, Z = x[2] + sk, far = 2 * rx + 1e-12;
    if (1 - X < -far || X - Y < -far || Y - Z < -far || Z < -far) return;
    double d[4][3], t[4], change = 0;
    for (int k = 0; k < 4; k++) {
        double s = 0;
        for (int i = 0; i < 3; i++) {
            d[k][i] = x[i] - corner[k][i] + k / 6.0;
            s += d[k][i] * d[k][i];
        }
        t[k] = fmax(0.5 - s, 0);
        /* the cell's largest t and s */
        const double r0 = fmax(sqrt(s) - rx, 0), r1 = fmin(sqrt(s) + rx, sqrt(0.5)), S = r1 * r1;
        const double T = fmax(0.5 - r0 * r0, 0), T2 = T * T, T3 = T2 * T;
        change += which == 0   ? T2 * T2 + 8 * T3 * S
                  : which == 1 ? 24 * T3 * r1 + 48 * T2 * S * r1
                               : 24 * T3 + 288 * T2 * S + 192 * T * S * S;
    }
    change *= 76.8 * ROOT2 * rx;
    for (int k = 0; k < 2; k++) {
        const double v = largest(&sets[k], d, t);
        if (1 - X >= 0 && X - Y >= 0 && Y - Z >= 0 && Z >= 0) {
            if (v > *seen) *seen = v;
            if (v > limit) state = 1;
        }
        if ((v + change) / sets[k].factor < limit) return;
        if (v + change >= limit) break; /* the fine set would not do either */
    }
    for (int k = 0; k < 8; k++) {
        const double c[3] = {x[0] + (k & 1 ? hx : -hx) / 2, x[1] + (k & 2 ? hx : -hx) / 2, x[2] + (k & 4 ? hx : -hx) / 2};
        visit(c, hx / 2, count, seen);
    }
}

int main(int argc, char **argv) {
    if (argc != 3) return 3;
    which = atoi(argv[1]);
    limit = atof(argv[2]);
    fill(&sets[0], COARSE);
    fill(&sets[1], FINE);
    /* the simplex lies within [-1/2, 1] per axis */
    enum { N = 16 };
    const double h = 0.75 / N;
#pragma omp parallel for schedule(dynamic, 1) reduction(+ : cells) reduction(max : best)
    for (int i = 0; i < N * N * N; i++) {
        const double c[3] = {-0.5 + h * (2 * (i % N) + 1), -0.5 + h * (2 * (i / N % N) + 1), -0.5 + h * (2 * (i / N / N) + 1)};
        visit(c, h, &cells, &best);
    }
    printf("%d %.6f %ld\n", which, best, cells);
    return state;
}
