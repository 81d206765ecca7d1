/*
 * scope_device.c - GPU check of the boxes that bound the next classification.
 *
 * Marches a case with moving bodies one step at a time.  After each step (two
 * solid half-steps) the scope that the device's classification left - every
 * body's node box and the box of the reconstructed nodes - must be the one
 * that a scan of the host's node flags over the whole interior gives.
 * Prints "ok <steps> <bodies that lost all their nodes>" or the first
 * difference and exits 1.
 *
 *   scope_device <case dir> <steps>
 */
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "artra_hip.h"
#include "solver.h"

static int Empty(const int box[DIMS][LIMIT])
{
    int empty = 0;
    for (int s = 0; s < DIMS; ++s) empty |= (box[s][MIN] >= box[s][MAX]);
    return empty;
}

static int Same(const int a[DIMS][LIMIT], const int b[DIMS][LIMIT])
{
    if (Empty(a) || Empty(b)) return Empty(a) && Empty(b);
    return 0 == memcmp(a, b, sizeof(int[DIMS][LIMIT]));
}

static int Differs(const char *what, int n, int step, const int got[DIMS][LIMIT], const int want[DIMS][LIMIT])
{
    if (Same(got, want)) return 0;
    printf("step %d: %s %d", step, what, n);
    for (int s = 0; s < DIMS; ++s) printf(" [%d %d) / [%d %d)", got[s][MIN], got[s][MAX], want[s][MIN], want[s][MAX]);
    printf("\n");
    return 1;
}

int main(int argc, char **argv)
{
    if (argc < 3) {
        fprintf(stderr, "usage: scope_device <case dir> <steps>\n");
        return 2;
    }
    const int steps = atoi(argv[2]);
    Time time;
    Space space;
    Model model;
    memset(&time, 0, sizeof time);
    memset(&space, 0, sizeof space);
    memset(&model, 0, sizeof model);
    ArtraHipSolver *s = NULL;
    if (artra_prepare_case(argv[1], &time, &space, &model) || artra_hip_attach(&space, &model, &s) ||
        artra_hip_treat_boundary(s, TO)) {
        fprintf(stderr, "%s\n", artra_hip_error());
        return 2;
    }
    for (int step = 1; step <= steps; ++step) {
        int done = 0;
        Real dt = 0.0;
        if (artra_hip_march(s, &time, 1, &done, &dt) || 1 != done) {
            fprintf(stderr, "step %d: %s\n", step, artra_hip_error());
            return 2;
        }
        ArtraGeometryScope want;
        if (artra_scope_init(&space, &want)) return 2;
        for (int n = 0; n < want.bodies; ++n) {
            if (Differs("body", n, step, (const int (*)[LIMIT])s->scope.extent[n], (const int (*)[LIMIT])want.extent[n]))
                return 1;
        }
        if (Differs("join", 0, step, (const int (*)[LIMIT])s->scope.join, (const int (*)[LIMIT])want.join)) return 1;
        artra_scope_free(&want);
    }
    int gone = 0;
    for (int n = 0; n < s->scope.bodies; ++n) gone += Empty((const int (*)[LIMIT])s->scope.extent[n]);
    artra_hip_detach(s);
    printf("ok %d %d\n", steps, gone);
    return 0;
}
