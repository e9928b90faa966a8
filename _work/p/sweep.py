"""sweep.py <family> : start's kernels against the present ones, graphs replayed in turn."""
import sys, importlib.util, statistics, math, random, time
sys.path.insert(0, '.')
import torch
def load(path, name):
    spec = importlib.util.spec_from_file_location(name, path)
    m = importlib.util.module_from_spec(spec); spec.loader.exec_module(m); return m
SO = '.cpython-310-x86_64-linux-gnu.so'
OLD = sys.argv[2] if len(sys.argv) > 2 else '_work/start'
S = load(f'{OLD}/xllm_service_amd/_ops{SO}', 'old._ops')
N = load(f'xllm_service_amd/_ops{SO}', 'new._ops')
SH = load(f'{OLD}/xllm_service_amd/_ops_hybrid{SO}', 'old._ops_hybrid')
NH = load(f'xllm_service_amd/_ops_hybrid{SO}', 'new._ops_hybrid')
assert S is not N and ('alt' in OLD or not hasattr(S,'linear_gated')) and hasattr(N,'linear_gated'), (S,N)
dev = 'cuda'
def graph(calls):
    for c in calls[:2]: c()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for c in calls: c()
    return g
def compare(name, a_calls, b_calls, out, reps=9):
    n = len(a_calls)
    ga, gb = graph(a_calls), graph(b_calls)
    ga.replay(); gb.replay(); torch.cuda.synchronize()
    ta, tb = [], []
    for _ in range(reps):
        for g, t in ((ga, ta), (gb, tb)):
            e0, e1 = torch.cuda.Event(True), torch.cuda.Event(True)
            e0.record(); g.replay(); e1.record(); torch.cuda.synchronize()
            t.append(e0.elapsed_time(e1) * 1e3 / n)
    a, b = statistics.median(ta), statistics.median(tb)
    print(f"{b/a:6.3f} {a:8.2f} {b:8.2f}  {name}", file=out, flush=True)
    if b / a > 1.02: print(f"{b/a:6.3f} {a:8.2f} {b:8.2f}  {name}", flush=True)
    del ga, gb
fam = sys.argv[1]
out = open(f'gpurun_out/sweep_{fam}.txt', 'w')
last = time.time()
def tick():
    global last
    if time.time() - last > 30: print('...', flush=True); last = time.time()
if fam in ('linear', 'bias'):
    NK = [(6144,2048),(8192,2048),(5120,2048),(7168,1024),(2048,2048),(3072,2048),(4096,2048),(2048,4096),(4096,4096),(6144,4096),(8192,4096),(28672,4096),(4096,14336),
          (4608,3584),(3584,3584),(37888,3584),(3584,18944),(14336,2048),(2304,768),(768,768),(3072,768),(768,3072),(32000,4096),
          (512,2048),(1024,1024),(1024,4096),(1536,2048),(12288,4096),(5120,5120),(2560,2560),(640,2560),(256,4096)]
    if fam == 'bias': NK = [(2048,2048),(4608,3584),(3072,2048),(6144,4096),(2304,768),(768,3072),(8192,4096),(1024,1024)]
    Ms = [1,2,4,6,8,10,12,16,20,24,28,32,40,48,56,64,80,96,128,160,192,224,256,300,384,512,768,1024,1536,2048]
    for n, k in NK:
        copies = int(max(6, min(48, (512 << 20) // (2*n*k))))
        W = [torch.randn(n, k, device=dev, dtype=torch.bfloat16) for _ in range(copies)]
        bias = torch.randn(n, device=dev, dtype=torch.bfloat16) if fam == 'bias' else None
        for m in Ms:
            x = torch.randn(m, k, device=dev, dtype=torch.bfloat16)
            ca = [lambda w=w: S.linear(x, w, bias) for w in W]
            cb = [lambda w=w: N.linear(x, w, bias) for w in W]
            compare(f'{fam} M {m} N {n} K {k}', ca, cb, out); tick()
        del W; torch.cuda.empty_cache()
if fam == 'rand':
    rng = random.Random(int(sys.argv[3]) if len(sys.argv) > 3 else 1)
    ex = lambda a,b: math.exp(rng.uniform(math.log(a), math.log(b)))
    for _ in range(70):
        n = max(16, int(ex(128, 33000))//64*64); k = max(128, int(ex(256, 16000))//128*128)
        if n*k > 140e6: continue
        copies = int(max(6, min(48, (512 << 20) // (2*n*k))))
        W = [torch.randn(n, k, device=dev, dtype=torch.bfloat16) for _ in range(copies)]
        for m in [max(1, int(ex(1, 2300))) for _ in range(7)]:
            x = torch.randn(m, k, device=dev, dtype=torch.bfloat16)
            compare(f'rand M {m} N {n} K {k}', [lambda w=w: S.linear(x, w, None) for w in W], [lambda w=w: N.linear(x, w, None) for w in W], out, 11); tick()
        del W; torch.cuda.empty_cache()
def pages(lens, wide=0):
    need = [-(-n // 16) for n in lens]; tot = sum(need) + 7
    order = torch.randperm(tot, device=dev).int()
    t = torch.zeros(len(lens), max(max(need), wide), dtype=torch.int32, device=dev); at = 0
    for i, n in enumerate(need): t[i,:n] = order[at:at+n]; at += n
    return t, tot
i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
def prefill(name, H, G, D, new, old, wide=0):
    T = sum(new); lens = [a+b for a,b in zip(new, old)]
    t, tot = pages(lens, wide)
    calls = []
    cu = [0]
    for n in new: cu.append(cu[-1]+n)
    cu, sl = i32(cu), i32(lens)
    copies = 3
    for _ in range(copies):
        q = torch.randn(T, H, D, device=dev).bfloat16()
        k, v = (torch.randn(tot, G, 16, D, device=dev).bfloat16() for _ in 'kv')
        o = torch.empty_like(q)
        calls.append((o, q, k, v))
    ca = [lambda c=c: S.paged_attn_prefill(*c, t, cu, sl, D**-0.5) for c in calls] * 4
    cb = [lambda c=c: N.paged_attn_prefill(*c, t, cu, sl, D**-0.5) for c in calls] * 4
    compare(f'prefill {H}/{G}x{D} {name} wide {wide}', ca, cb, out); tick()
if fam == 'prefill':
    heads = [(32,8,128),(28,4,128),(16,4,128),(8,1,128),(64,8,128),(12,12,64),(32,32,128),(4,2,64)]
    rng = random.Random(5)
    for H, G, D in heads:
        for new, old in [([1],[100]),([16],[0]),([16],[500]),([17],[2000]),([32],[120]),([50],[1000]),([64],[0]),([64],[64]),([100],[0]),([100],[800]),([100],[1900]),
                         ([128],[0]),([150]*2,[0]*2),([200],[0]),([200],[300]),([200],[1500]),([256],[0]),([300],[0]),([300],[700]),([400],[0]),([512],[0]),([512],[512]),([700],[0]),
                         ([1000],[0]),([1000],[1000]),([1024],[0]),([1500],[0]),([2000],[0]),([2000,2500],[0,0]),([2048]*2,[0]*2),([2500],[0]),([3000],[0]),([4096],[0]),([4096],[4000]),([8192],[0]),
                         ([16]*8,[200]*8),([20]*16,[500]*16),([64]*8,[0]*8),([64]*8,[1000]*8),([512]*8,[0]*8),([500]*7+[2100],[0]*8),([1024]*4,[0]*4),([256]*16,[0]*16),
                         ([256]*16,[1900]*16),([100]*40,[2000]*40),([1]*60+[500],[300]*61),([2200]+[100]*20,[0]*21),([4200,100],[0,3000]),([3000,2000],[0,3000]),([600]*4,[600]*4),([800]*3,[1300]*3)]:
            if sum(new)*H*(sum(old)/len(old)+sum(new)/len(new))*D*2 > 4e12: continue
            prefill(f'{new if len(new)<4 else str(len(new))+"x"+str(new[0])+".."+str(new[-1])} behind {old if len(old)<4 else old[0]}', H, G, D, new, old)
        for new, old, wide in [([100],[100],256),([300],[0],128),([300],[0],512),([30],[60],64),([2500],[0],300),([20]*10,[30]*10,100)]:
            prefill(f'{new} behind {old}', H, G, D, new, old, wide)
        for i in range(25):
            n = rng.choice([1,1,2,3,5,8]); 
            new = [int(math.exp(rng.uniform(math.log(16), math.log(2500)))) for _ in range(n)]
            old = [int(math.exp(rng.uniform(math.log(16), math.log(3000)))) if rng.random()<.6 else 0 for _ in range(n)]
            if sum(new) > 8192: continue
            prefill(f'{new} behind {old}', H, G, D, new, old)
if fam == 'latent':
    rng = random.Random(7)
    def lat(name, heads, tail, lens, window=0, wide=0):
        t, tot = pages(lens, wide); W = 512 + tail
        cs = []
        for _ in range(3):
            cs.append((torch.empty(len(lens), heads, 512, device=dev), torch.randn(len(lens), heads, W, device=dev).bfloat16(), torch.randn(tot, 16, W, device=dev).bfloat16()))
        sl = i32(lens)
        ca = [lambda c=c: SH.latent_attn(*c, t, None, sl, 192**-0.5, 512, window) for c in cs]*4
        cb = [lambda c=c: NH.latent_attn(*c, t, None, sl, 192**-0.5, 512, window) for c in cs]*4
        compare(f'latent heads {heads} tail {tail} win {window} {name} wide {wide}', ca, cb, out); tick()
    for heads, tail in [(16,64),(16,0),(32,64),(128,64),(20,64)]:
        for n in [1,2,4,8,12,16,20,23,24,28,32,40,43,48,64,80,85,86,90,100,128,160,200,256,257,300]:
            for L in [30,100,300,700,1000,1024,2000,4000]:
                if n*L > 400000 or n*heads>5000: continue
                lat(f'{n} x {L}', heads, tail, [L]*n)
            for hi in (900, 4000):
                ls = [int(math.exp(rng.uniform(math.log(50), math.log(hi)))) for _ in range(n)]
                lat(f'{n} x 50-{hi}', heads, tail, ls)
            lat(f'{n} x 2000', heads, tail, [2000]*n, 512)
            lat(f'{n} x 500', heads, tail, [500]*n, 0, 256)
if fam == 'decay':
    for H, D in [(16,128),(32,128),(8,64),(64,128)]:
        for new in [[17],[32],[64],[100],[128],[129],[300],[700],[1000],[2000],[4000],[8000],[100]*8,[300]*4,[40]*30,[700,2000,1300],[1,5,900],[20]*100]:
            for ctx in (0, 64):
                T = sum(new)
                rows = torch.randn(T, 4*H*D, device=dev).bfloat16()
                q,k,v = (rows[:, i*H*D:(i+1)*H*D] for i in range(3))
                dec = torch.tensor([1-2.0**-(2+6*h/max(H-1,1)) for h in range(H)], device=dev)
                st = torch.randn(len(new)+1, H, D, D, device=dev); sl = torch.arange(len(new), device=dev).int()
                cu=[0]
                for n in new: cu.append(cu[-1]+n)
                cu, cx = i32(cu), i32([ctx]*len(new))
                o = torch.empty(T, H, D, device=dev)
                ca = [lambda: SH.decay_attn(o,q,k,v,dec,st,sl,cu,cx,max(new))]*8
                cb = [lambda: NH.decay_attn(o,q,k,v,dec,st,sl,cu,cx,max(new))]*8
                compare(f'decay {H}x{D} {new if len(new)<4 else str(len(new))+"x"+str(new[0])} ctx {ctx}', ca, cb, out); tick()
print('done', fam)
if fam == 'rest':
    for n, k in [(512,2304),(512,3072),(768,2304),(768,2560),(768,3072),(768,4096),(512,4096),(1024,3072),(2560,2560),(2304,2560),(2048,2560),(2816,2560),(3072,2560)]:
        copies = int(max(6, min(48, (512 << 20) // (2*n*k))))
        W = [torch.randn(n, k, device=dev, dtype=torch.bfloat16) for _ in range(copies)]
        for m in [260,288,300,320,350,384,400,448,512,640,768,1000] if n < 2000 else [300,320,384,400]:
            x = torch.randn(m, k, device=dev, dtype=torch.bfloat16)
            compare(f'rest M {m} N {n} K {k}', [lambda w=w: S.linear(x, w, None) for w in W], [lambda w=w: N.linear(x, w, None) for w in W], out, 15); tick()
        del W; torch.cuda.empty_cache()
    for H, G in [(64,8),(32,8),(32,32),(8,1)]:
        for new, old in [([800]*3,[1300]*3),([1000]*3,[1300]*3),([600]*4,[1300]*4),([800]*3,[0]*3),([1500],[1300]),([2000],[0]),([2500],[0]),([17],[2000]),([17],[1000]),([30],[2000]),([17]*2,[2000]*2)]:
            prefill(f'{new} behind {old}', H, G, 128, new, old)
    print('done rest')
if fam == 'rest2':
    seen = set()
    for H, G in [(32,8),(64,8),(32,32),(28,4),(16,2)]:
        for w in [440,470,512,516,540,580,620,640,660,700,740,770,800,850,900,1030,1060,1100]:
            T = int(w / G * 256 / (H // G))
            for n, old in [(1,0),(1,.3),(1,1),(1,2.5),(2,0),(2,.7),(3,1),(3,2.5),(2,6)]:
                new = [T // n] * n
                if old * new[0] + new[0] < 2048 or T < 256 * n or (old+.5)*T*T/n*H*512 > 6e12: continue
                prefill(f'w {w} n {n} old {old} {new} behind {int(new[0]*old)}', H, G, 128, new, [int(new[0]*old)]*n)
    for H, G in [(32,32),(16,16),(8,8),(32,8),(16,4),(64,64),(28,4),(64,8)]:
        for new in [17, 30, 45, 60, 100]:
            for n in [1, 2, 4]:
                for old in [1000, 1250, 1400, 1510, 1600, 1750, 1930]:
                    prefill(f's {new}x{n} behind {old}', H, G, 128, [new]*n, [old]*n)
    print('done rest2')
if fam == 'rest3':
    rng = random.Random(11)
    done = 0
    while done < 150:
        H, G = rng.choice([(32,8),(64,8),(32,32),(28,4),(16,2)])
        n = rng.choice([2,2,3,4,5,6,8,12])
        new = [int(math.exp(rng.uniform(math.log(60), math.log(6000)))) for _ in range(n)]
        old = [int(math.exp(rng.uniform(math.log(60), math.log(6000)))) if rng.random()<.5 else 0 for _ in range(n)]
        T = sum(new); w = T*H/256; K = max(a+b for a,b in zip(new,old))
        if w < 430 or w > 1150 or K < 2048 or T < 256*n: continue
        done += 1
        prefill(f'w {w:.0f} n {n} K {K} avg {T//n} eq {-(-T*(H//G)//(n*256))*n*G} {new} behind {old}', H, G, 128, new, old)
    print('done rest3')
if fam == 'rest4':
    for H, G in [(32,8),(64,8),(32,32),(28,4),(16,2)]:
        for w in [440,470,512,516,540,580,640,660,700,770,850,900,1030,1100]:
            T = int(w / G * 256 / (H // G))
            for n, old in [(1,0),(1,.3),(1,1),(2,0),(2,.7),(3,1),(3,2.5)]:
                new = [T // n] * n
                if old * new[0] + new[0] < 2048 or T < 256 * n or (old+.5)*T*T/n*H*512 > 3e12: continue
                prefill(f'w {w} n {n} old {old} {new} behind {int(new[0]*old)}', H, G, 128, new, [int(new[0]*old)]*n)
    print('done rest4')
if fam == 'rest5':
    for H, G in [(12,12),(4,2),(16,16),(32,8),(16,2)]:
        for new in [17, 30, 60, 100]:
            for n in [1, 2, 4]:
                for old in [200, 300, 400, 500, 600, 700, 800, 920]:
                    prefill(f's {new}x{n} behind {old}', H, G, 64, [new]*n, [old]*n)
    for H, G in [(32,32),(16,16),(8,8),(32,8),(16,4),(28,4),(64,8)]:
        for new in [17, 30, 45, 60, 100]:
            for n in [1, 4]:
                for old in [200,300,400, 500, 700, 850, 920,1000, 1400, 1510, 1600, 1750, 1930]:
                    prefill(f't {new}x{n} behind {old}', H, G, 128, [new]*n, [old]*n)
    print('done rest5')
if fam == 'rest6':
    for n, k in [(512,2560),(512,3072),(768,2560),(768,3072),(768,4096),(512,4096),(576,4096),(896,3072),(960,3584)]:
        copies = int(max(6, min(48, (512 << 20) // (2*n*k))))
        W = [torch.randn(n, k, device=dev, dtype=torch.bfloat16) for _ in range(copies)]
        for m in [260,300,320,350,384,448,512,576,640,1000]:
            x = torch.randn(m, k, device=dev, dtype=torch.bfloat16)
            compare(f'rest M {m} N {n} K {k}', [lambda w=w: S.linear(x, w, None) for w in W], [lambda w=w: N.linear(x, w, None) for w in W], out, 15); tick()
        del W; torch.cuda.empty_cache()
    print('done rest6')
