/*
 * lm_shapes.c — which prompt shapes are kept as captured graphs (host only).
 *
 * A prompt's length is often its own, so a shape is launched directly the first
 * time and captured when it comes again.  With every graph in use, a shape takes
 * the least recently used one's place only if that one has not been used since
 * the shape's own last time: more shapes in rotation than graphs then keep the
 * graphs of some, which replay, and launch the others directly, where replacing
 * a graph at each call would capture at each call.
 */
#include "lm_internal.h"

static int same(const LMShape *a, int R, int S, int all)
{
    return a->used && a->R == R && a->S == S && a->all == all;
}

static int oldest(const LMShape *a, int n)
{
    int k = 0;
    for (int i = 1; i < n; i++)
        if (a[i].used < a[k].used) k = i;   /* (an empty one is 0) */
    return k;
}

int lmh_shape_use(LMShapes *t, int R, int S, int all, int *slot)
{
    const unsigned long now = ++t->calls;
    for (int k = 0; k < LM_SHAPE_GRAPHS; k++)
        if (same(&t->graph[k], R, S, all)) {
            t->graph[k].used = now;
            *slot = k;
            return LM_SHAPE_REPLAY;
        }
    const LMShape me = {R, S, all, now};
    for (int i = 0; i < LM_SHAPE_SEEN; i++) {
        if (!same(&t->seen[i], R, S, all)) continue;
        const unsigned long before = t->seen[i].used;
        const int k = oldest(t->graph, LM_SHAPE_GRAPHS);
        if (t->graph[k].used > before) {
            t->seen[i].used = now;
            return LM_SHAPE_DIRECT;
        }
        t->seen[i].used = 0;
        t->graph[k] = me;
        *slot = k;
        return LM_SHAPE_CAPTURE;
    }
    t->seen[oldest(t->seen, LM_SHAPE_SEEN)] = me;
    return LM_SHAPE_DIRECT;
}
